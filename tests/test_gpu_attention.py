"""GPU parity of the attention kernel (csrc/attention.cpp): key counts off its
16-key blocks, query rows off its 16-row tiles, every split of rows and columns
over waves, orders of the grid, part of an array, buffers off its alignment.

Bar: the f32 softmax's 1e-5 (relative, Frobenius) against the oracle.
"""

from __future__ import annotations

import numpy as np
import pytest

import xtile_amd as xt
from oracle import f32_to_bf16_bits
from tests.conftest import oracle_threads
from tests.gpu_util import frob_rel, kernels_of, run_gpu, run_oracle, to_device
from xtile_amd import kernels as K

pytestmark = pytest.mark.gpu

_XT = {"f16": xt.float16, "bf16": xt.bfloat16}


def _inputs(seed, q, k, v, dt):
    rng = np.random.default_rng(seed)
    a, b = rng.normal(0, 0.5, q).astype(np.float32), rng.normal(0, 0.5, k).astype(np.float32)
    a, b = (a.astype(np.float16), b.astype(np.float16)) if dt == "f16" else (f32_to_bf16_bits(a), f32_to_bf16_bits(b))
    return [a, b, rng.normal(0, 1, v).astype(np.float32), np.full(q, np.nan, np.float32)]


def _check(cuda, m, bufs, dt, case):
    assert " attention waves=" in xt.plan(m)["kernel"]
    got = run_gpu(m, bufs, [dt, dt, "f32", "f32"], cuda, case=case, kernels=["xt_attend"])[3]
    want = run_oracle(m, bufs, oracle_threads())[3]
    assert frob_rel(got, want) <= 1e-5


@pytest.mark.parametrize(
    "heads,nq,nk,d,tq,dt",
    [(1, 1, 1, 32, 1, "f16"),         # one query, one key
     (3, 13, 33, 32, 13, "bf16"),     # keys and rows past whole blocks
     (2, 40, 15, 64, 20, "f16"),      # fewer keys than a block
     (10, 48, 40, 64, 16, "f16"),     # four waves share the columns of 16 rows
     (200, 32, 72, 64, 32, "bf16"),   # 2 row tiles x 4 column shares
     (200, 70, 65, 128, 35, "f16"),   # 128 columns, rows past the last tile
     (400, 144, 16, 32, 16, "f16"),   # whole rows a wave, uneven tiles a workgroup
     (300, 272, 160, 128, 16, "bf16"),  # several tiles a workgroup
     (2, 32, 496, 32, 16, "f16")],    # the most keys
)
def test_attention(cuda, heads, nq, nk, d, tq, dt):
    m = K.attention(heads, nq, nk, d, tq, qk=_XT[dt])
    _check(cuda, m, _inputs(nq + nk, (heads, nq, d), (heads, nk, d), (heads, nk, d), dt), dt,
           f"attention {heads}x{nq}x{nk}x{d} tq={tq} {dt}")


@xt.kernel
def _heads_first(q, k, v, o, tq, d, nk):
    """Heads along axis 0, query tiles along axis 2, no shared loads."""
    h = xt.bid(0)
    i = xt.bid(2)
    qt = xt.reshape(xt.load(q, index=(h, i, 0), shape=(1, tq, d)), shape=(tq, d))
    kt = xt.load(k, index=(h, 0, 0), shape=(1, nk, d))
    vt = xt.reshape(xt.load(v, index=(h, 0, 0), shape=(1, nk, d)), shape=(nk, d))
    s = xt.matmul(qt, xt.reshape(xt.transpose(kt), shape=(d, nk)))
    p = xt.exp(xt.sub(s, xt.max(s, axis=1)))
    p = xt.mul(p, xt.reciprocal(xt.sum(p, axis=1)))
    xt.store(o, index=(h, i, 0), tile=xt.reshape(xt.matmul(p, vt), shape=(1, tq, d)))


@xt.kernel
def _column_heads(q, k, v, o, tq, d, nk):
    """Heads are column groups of [rows, heads * d] arrays; keys are the second
    nk rows of theirs, and every query tile has keys of its own head only."""
    h = xt.bid(1)
    i = xt.bid(0)
    qt = xt.load(q, index=(i, h), shape=(tq, d))
    kt = xt.load(k, index=(1, h), shape=(nk, d))
    vt = xt.load(v, index=(1, h), shape=(nk, d))
    s = xt.matmul(qt, xt.reshape(xt.transpose(xt.reshape(kt, shape=(1, nk, d))), shape=(d, nk)))
    p = xt.exp(xt.sub(s, xt.max(s, axis=1)))
    p = xt.mul(p, xt.reciprocal(xt.sum(p, axis=1)))
    xt.store(o, index=(i, h), tile=xt.matmul(p, vt))


@xt.kernel
def _own_keys(q, k, v, o, tq, d, nk):
    """Keys move with the query tile: no two tiles share a workgroup."""
    i = xt.bid(0)
    qt = xt.load(q, index=(i, 0), shape=(tq, d))
    kt = xt.load(k, index=(i, 0), shape=(nk, d))
    vt = xt.load(v, index=(i, 0), shape=(nk, d))
    s = xt.matmul(qt, xt.reshape(xt.transpose(xt.reshape(kt, shape=(1, nk, d))), shape=(d, nk)))
    p = xt.exp(xt.sub(s, xt.max(s, axis=1)))
    p = xt.mul(p, xt.reciprocal(xt.sum(p, axis=1)))
    xt.store(o, index=(i, 0), tile=xt.matmul(p, vt))


@pytest.mark.parametrize("form", ["heads_first", "column_heads", "own_keys"])
def test_orders_and_strides(cuda, form):
    tq, d, nk = 24, 64, 56
    if form == "heads_first":
        fn, q, k, grid = _heads_first, (5, 3 * tq, d), (5, nk, d), (5, 1, 3)
    elif form == "column_heads":
        fn, q, k, grid = _column_heads, (3 * tq, 4 * d), (2 * nk, 4 * d), (3, 4, 1)
    else:
        fn, q, k, grid = _own_keys, (4 * tq, d), (4 * nk, d), (4, 1, 1)
    m = xt.convert(fn, args=(xt.Array(q, xt.float16), xt.Array(k, xt.float16), xt.Array(k, xt.float32),
                             xt.Array(q, xt.float32), tq, d, nk), grid=grid)
    _check(cuda, m, _inputs(9, q, k, k, "f16"), "f16", form)


def test_infinite_scores(cuda):
    """A row whose scores hold an infinity is NaN, one with a -inf key gives that
    key no weight, as on the oracle."""
    m = K.attention(1, 32, 40, 32, 32)
    bufs = _inputs(3, (1, 32, 32), (1, 40, 32), (1, 40, 32), "f16")
    bufs[0][0, 3, 0] = np.inf
    bufs[0][0, 5, :] = 0
    bufs[0][0, 5, 1] = 1
    bufs[1][0, 7, 1] = -np.inf
    bufs[1][0, :, 0] = np.abs(bufs[1][0, :, 0]) + np.float16(0.1)
    bufs[0][0, :, 1] = np.abs(bufs[0][0, :, 1]) + np.float16(0.1)
    got = run_gpu(m, bufs, ["f16", "f16", "f32", "f32"], cuda, case="infinite scores")[3]
    want = run_oracle(m, bufs, 1)[3]
    assert np.isnan(want[0, 3]).all() and np.isfinite(want[0, 5]).all()
    np.testing.assert_allclose(got, want, rtol=0, atol=2e-5)


@pytest.mark.parametrize("off", [1, 4])
def test_buffers_off_the_alignment(cuda, off):
    """Buffers 4 elements past an aligned address run the staged kernel, 1
    element past its scalar variant."""
    import torch

    m = K.attention(2, 64, 48, 64, 32)
    bufs = _inputs(4, (2, 64, 64), (2, 48, 64), (2, 48, 64), "f16")
    dev = []
    for x, dt in zip(bufs, ("f16", "f16", "f32", "f32")):
        t = to_device(x, dt, cuda)
        flat = torch.zeros(x.size + 8, dtype=t.dtype, device=cuda)
        flat[off : off + x.size] = t.reshape(-1)
        dev.append(flat[off : off + x.size].view(x.shape))
    print(f"[gpu] attention, buffers {off} elements off", flush=True)
    assert kernels_of(m, dev) == ["xt_fused"]
    xt.launch(m, *dev)
    torch.cuda.synchronize()
    assert frob_rel(dev[3].cpu().numpy(), run_oracle(m, bufs, 1)[3]) <= 1e-5


@pytest.mark.parametrize("how", ["one memref", "one tensor"])
def test_result_over_the_values(cuda, how):
    """The result stored over V, a Block's own tile each: as one memref of the
    program, and as one tensor passed for both.  Either runs one workgroup a
    Block, which has V in LDS before it stores."""
    import torch

    t, n, d = 128, 64 * 128, 64
    m = xt.convert(_own_keys, args=(xt.Array((n, d), xt.float16), xt.Array((n, d), xt.float16), xt.Array((n, d), xt.float32),
                                    xt.Array((n, d), xt.float32), t, d, t), grid=(n // t, 1, 1))
    bufs = _inputs(11, (n, d), (n, d), (n, d), "f16")
    want = run_oracle(m, bufs, oracle_threads())[3]
    dev = [to_device(x, dt, cuda) for x, dt in zip(bufs, ("f16", "f16", "f32", "f32"))]
    print(f"[gpu] attention over its values, {how}", flush=True)
    if how == "one tensor":
        assert kernels_of(m, dev) == ["xt_attend"]
    if how == "one memref":
        over_v = str(m).replace("%matmul2, %output,", "%matmul2, %input3,")
        assert over_v != str(m) and " attention waves=" not in xt.plan(xt.parse(over_v))["kernel"]
        xt.launch(xt.parse(over_v), *dev)
    else:
        xt.launch(m, dev[0], dev[1], dev[2], dev[2])
    torch.cuda.synchronize()
    assert frob_rel(dev[2].cpu().numpy(), want) <= 1e-5
    if how == "one tensor":
        assert kernels_of(m, [dev[0], dev[1], dev[2], dev[2]]) == ["xt_fused"]
