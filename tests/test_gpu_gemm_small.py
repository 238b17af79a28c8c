"""GPU parity of the GEMM kernels where their tiles do not divide the product:
gemm_small.hip's 32- and 64-wide tiles (LDS DMA, and the register path for
sizes and alignments DMA does not take) and the DMA kernel's edge tiles,
against float64 products (oracle.closed_form.matmul).

Tolerance: each of K f32 additions rounds by at most 2^-24 of its partial sum;
the signs are random, so the result is off by about sqrt(K) 2^-24 of its norm,
and the bar is four times that.  i8 results are whole numbers and equal.
"""

from __future__ import annotations

import numpy as np
import pytest

import xtile_amd as xt
from oracle import bf16_bits_to_f32, closed_form, f32_to_bf16_bits
from tests.conftest import oracle_threads
from tests.gpu_util import frob_rel, kernels_of, run_gpu, run_oracle, to_device
from tests.test_plan import i8_over
from xtile_amd import kernels as K

pytestmark = pytest.mark.gpu


def _narrow(rng, shape, dt):
    x = rng.uniform(-1, 1, shape).astype(np.float32)
    return x.astype(np.float16) if dt == "f16" else f32_to_bf16_bits(x)


def _wide(x):
    return (bf16_bits_to_f32(x) if x.dtype == np.uint16 else x).astype(np.float64)


def _bar(k):
    return 4 * np.sqrt(k) * 2.0**-24


_ELEM = {"f16": 0, "bf16": 1, "i8": 2}


def _small(dt, bm, bn, load, out_i8=0):
    return [f"gemm_small_kernel<{_ELEM[dt]}, {out_i8}, {bm}, {bn}, {load}>"]


def _edge(dt, t, epilogue=0, out_i8=0):
    waves = 8 if t == 256 else 4
    return [f"gemm_dma_kernel<{_ELEM[dt]}, 4, {out_i8}, {epilogue}, {waves}, 0, {t}, {t}, 1>"]


_DMA, _REGS = 0, 1
_SPLIT = ["gemm_zero_kernel", "gemm_dma_kernel<0, 4, 0, 0, 4, 1, 128, 128, 0>"]


@pytest.mark.parametrize(
    "dt,m,n,k,tm,tn,family,kernels",
    [("f16", 40, 40, 72, 40, 40, "staged", _small("f16", 32, 32, _DMA)),        # K tail of one chunk
     ("bf16", 96, 200, 520, 48, 40, "staged", _small("bf16", 32, 32, _DMA)),    # N's last tile 8 wide
     ("f16", 8, 8, 8, 8, 8, "staged", _small("f16", 32, 32, _DMA)),             # the smallest DMA product
     ("bf16", 26, 65, 61, 13, 13, "staged", _small("bf16", 32, 32, _REGS)),     # one column in the last tile, odd K
     ("f16", 9, 9, 9, 9, 9, "staged", _small("f16", 32, 32, _REGS)),            # one more than a chunk
     ("f16", 95, 60, 146, 19, 20, "staged", _small("f16", 32, 32, _REGS)),      # several tiles
     ("bf16", 16, 7, 64, 16, 7, "staged", ["xt_fused"]),                        # N below a chunk
     ("f16", 1000, 1000, 1000, 40, 40, "staged", _small("f16", 64, 64, _DMA)),
     ("bf16", 999, 1001, 333, 37, 13, "staged", _small("bf16", 64, 64, _REGS)),
     ("f16", 1728, 330, 96, 36, 30, "staged", _small("f16", 64, 64, _REGS)),
     ("f16", 1260, 384, 72, 35, 48, "staged", _small("f16", 32, 64, _DMA)),
     ("bf16", 546, 528, 144, 26, 48, "staged", _small("bf16", 32, 64, _DMA)),
     ("f16", 2736, 68, 131, 48, 34, "staged", _small("f16", 32, 64, _REGS)),    # N's second tile 4 wide
     ("bf16", 912, 279, 92, 48, 31, "staged", _small("bf16", 32, 64, _REGS)),
     ("f16", 64, 64, 64, 64, 64, "gemm", _small("f16", 32, 32, _DMA)),          # fewer stages than waves
     ("bf16", 64, 320, 640, 64, 64, "gemm", _small("bf16", 32, 32, _DMA)),
     ("f16", 192, 1088, 4160, 64, 64, "gemm", _small("f16", 32, 32, _DMA)),
     ("f16", 1024, 1024, 1024, 128, 128, "gemm", _small("f16", 64, 64, _DMA)),
     ("f16", 2880, 512, 640, 64, 64, "gemm", _edge("f16", 128)),                # M edge
     ("bf16", 2112, 4160, 320, 64, 64, "gemm", _edge("bf16", 128)),             # M and N edges
     ("f16", 256, 512, 8192, 128, 64, "gemm", _SPLIT),                          # 8 tiles in 16 K ranges
     ("f16", 256, 256, 5376, 64, 64, "gemm", _SPLIT),
     ("f16", 256, 256, 2560, 64, 64, "gemm", _small("f16", 32, 32, _DMA)),
     ("f16", 1600, 6656, 512, 64, 128, "gemm", _edge("f16", 256)),              # M edge
     ("bf16", 4864, 2112, 256, 128, 64, "gemm", _edge("bf16", 256))],           # N edge
)
def test_products_no_tile_divides(cuda, dt, m, n, k, tm, tn, family, kernels):
    mod = (K.matmul_f16 if dt == "f16" else K.matmul_bf16)(m, n, k, tm, tn)
    assert xt.plan(mod)["kernel"].startswith(family)
    rng = np.random.default_rng(m + n + k)
    a, b = _narrow(rng, (m, k), dt), _narrow(rng, (k, n), dt)
    got = run_gpu(mod, [a, b, np.full((m, n), np.nan, np.float32)], [dt, dt, "f32"], cuda, case=f"{dt} {m}x{n}x{k}",
                  kernels=kernels)[2]
    assert frob_rel(got, closed_form.matmul(_wide(a), _wide(b))) <= _bar(k)


@pytest.mark.parametrize(
    "m,n,k,tm,tn,kernels",
    [(48, 40, 72, 16, 8, _small("i8", 32, 32, _REGS, 1)), (33, 51, 49, 33, 17, _small("i8", 32, 32, _REGS, 1)),
     (64, 128, 128, 64, 64, _small("i8", 32, 32, _DMA, 1)), (32, 65, 16, 16, 13, _small("i8", 32, 32, _REGS, 1)),
     (128, 1088, 4096, 64, 64, _small("i8", 32, 32, _DMA, 1)), (576, 512, 256, 64, 128, _small("i8", 32, 64, _DMA, 1)),
     (256, 2880, 256, 128, 64, _small("i8", 64, 64, _DMA, 1)), (448, 3072, 256, 64, 128, _edge("i8", 128, 1, 1)),
     (2112, 2240, 256, 64, 64, _edge("i8", 256, 1, 1))],
)
def test_i8_epilogue_products_no_tile_divides(cuda, m, n, k, tm, tn, kernels):
    """* scale + bias, astype(int8): the oracle's bytes."""
    mod = K.matmul_i8(m, n, k, tm, tn)
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    b = rng.integers(-128, 128, (k, n), dtype=np.int8)
    s = (rng.uniform(0.5, 2.0, (1, n)) / (np.sqrt(k) * 100)).astype(np.float32)
    bias = rng.uniform(-20, 20, (1, n)).astype(np.float32)
    bufs = [a, b, np.full((m, n), 99, np.int8), s, bias]
    got = run_gpu(mod, bufs, ["i8", "i8", "i8", "f32", "f32"], cuda, case=f"i8 {m}x{n}x{k}", kernels=kernels)[2]
    assert np.array_equal(got, run_oracle(mod, bufs, oracle_threads())[2])


@xt.kernel
def _scaled_kernel(a, b, out, scale, bias, tm, tn, tk):
    i = xt.bid(0)
    j = xt.bid(1)
    t = xt.matmul(xt.load(a, index=(i, 0), shape=(tm, tk)), xt.load(b, index=(0, j), shape=(tk, tn)))
    s = xt.load(scale, index=(0, j), shape=(1, tn))
    xt.store(out, index=(i, j), tile=t * s + xt.load(bias, index=(0, j), shape=(1, tn)))


@pytest.mark.parametrize(
    "dt,m,n,k,tm,tn,kernels",
    [("f16", 80, 72, 104, 40, 24, _small("f16", 32, 32, _DMA)),
     ("bf16", 26, 65, 61, 13, 13, _small("bf16", 32, 32, _REGS)),   # one column in the last tile
     ("f16", 1000, 600, 200, 40, 40, _small("f16", 64, 64, _DMA)),
     ("i8", 99, 85, 50, 33, 17, _small("i8", 32, 32, _REGS)),
     ("f16", 2880, 512, 640, 64, 64, _edge("f16", 128, 1)),         # M edge
     ("bf16", 4864, 2112, 256, 128, 64, _edge("bf16", 256, 1))],    # N edge
)
def test_f32_results_with_scale_and_bias(cuda, dt, m, n, k, tm, tn, kernels):
    """(a @ b) * scale + bias as f32: the product's bar, and a rounding each of the
    scaling and the sum."""
    e = {"f16": xt.float16, "bf16": xt.bfloat16, "i8": xt.int8}[dt]
    row = xt.Array((1, n), xt.float32)
    mod = xt.convert(_scaled_kernel, args=(xt.Array((m, k), e), xt.Array((k, n), e), xt.Array((m, n), xt.float32), row, row,
                                          tm, tn, k), grid=(m // tm, n // tn, 1))
    rng = np.random.default_rng(m + n + k)
    if dt == "i8":
        a, b = rng.integers(-128, 128, (m, k), dtype=np.int8), rng.integers(-128, 128, (k, n), dtype=np.int8)
    else:
        a, b = _narrow(rng, (m, k), dt), _narrow(rng, (k, n), dt)
    s, bias = (rng.uniform(0.5, 2, (1, n)).astype(np.float32) for _ in range(2))
    bufs = [a, b, np.full((m, n), np.nan, np.float32), s, bias]
    got = run_gpu(mod, bufs, [dt, dt, "f32", "f32", "f32"], cuda, case=f"{dt} {m}x{n}x{k} * s + b", kernels=kernels)[2]
    scaled = closed_form.matmul(_wide(a), _wide(b)) * s.astype(np.float64)
    want = scaled + bias.astype(np.float64)
    assert frob_rel(got, want) <= (_bar(k) + 2.0**-24) * np.linalg.norm(scaled) / np.linalg.norm(want) + 2.0**-24


@xt.kernel
def _part_kernel(a, b, out, tm, tn, tk):
    i = xt.bid(0)
    j = xt.bid(1)
    x = xt.load(a, index=(i, 1), shape=(tm, tk))
    w = xt.load(b, index=(1, j), shape=(tk, tn), shared=1)
    xt.store(out, index=(i, j), tile=xt.matmul(x, w))


@pytest.mark.parametrize("tm,tn,k", [(24, 40, 96), (20, 15, 33)])
def test_product_of_part_of_its_arrays(cuda, tm, tn, k):
    """A's second K columns, B's second K rows and half of B's and C's columns:
    origins, pitches and a region narrower than its arrays.  The rest of C
    stays as it was."""
    m, n = 3 * tm, 5 * tn
    mod = xt.convert(_part_kernel, args=(xt.Array((m, 2 * k), xt.float16), xt.Array((2 * k, 2 * n), xt.float16),
                                        xt.Array((m, 2 * n), xt.float32), tm, tn, k), grid=(3, 5, 1))
    assert xt.plan(mod)["kernel"].startswith("staged") and " gemm k=" in xt.plan(mod)["kernel"]
    rng = np.random.default_rng(7)
    a, b = _narrow(rng, (m, 2 * k), "f16"), _narrow(rng, (2 * k, 2 * n), "f16")
    c = np.full((m, 2 * n), 5.0, np.float32)
    got = run_gpu(mod, [a, b, c], ["f16", "f16", "f32"], cuda, case=f"part {tm}x{tn}x{k}")[2]
    assert frob_rel(got[:, :n], closed_form.matmul(_wide(a[:, k:]), _wide(b[k:, :n]))) <= _bar(k)
    assert np.all(got[:, n:] == 5.0)


def test_buffers_off_the_vector_alignment(cuda):
    """A, B and C one element past an aligned address: the register path, and
    element stores."""
    import torch

    m = n = k = 80
    mod = K.matmul_f16(m, n, k, 40, 40)
    rng = np.random.default_rng(8)
    a, b = _narrow(rng, (m, k), "f16"), _narrow(rng, (k, n), "f16")

    def shifted(x, dt):
        flat = torch.zeros(x.size + 1, dtype=dt, device=cuda)
        flat[1:] = to_device(x, "f16" if dt == torch.float16 else "f32", cuda).reshape(-1)
        return flat[1:].view(x.shape)

    dev = [shifted(a, torch.float16), shifted(b, torch.float16), shifted(np.zeros((m, n), np.float32), torch.float32)]
    print("[gpu] unaligned buffers", flush=True)
    assert kernels_of(mod, dev) == _small("f16", 32, 32, _REGS)
    xt.launch(mod, *dev)
    torch.cuda.synchronize()
    assert frob_rel(dev[2].cpu().numpy(), closed_form.matmul(_wide(a), _wide(b))) <= _bar(k)


@pytest.mark.parametrize("how", ["one memref", "one tensor"])
@pytest.mark.parametrize(
    "operand,blocks,t,n,kernel",
    [("a", 25, 40, 100, "xt_fused"), ("a", 64, 24, 132, "xt_fused"), ("b", 9, 40, 100, "xt_fused"),
     ("a", 8, 128, 128, "gemm_dma_kernel<2, 4, 1, 1, 4, 0, 128, 128, 0>"),
     ("a", 6, 64, 256, "gemm_dma_kernel<2, 4, 1, 1, 4, 0, 128, 256, 0>"),   # two Blocks a tile
     ("a", 5, 192, 128, "gemm_dma_kernel<2, 4, 1, 1, 4, 0, 128, 128, 1>"),  # the last tile half past M
     ("b", 7, 128, 128, "gemm_dma_kernel<2, 4, 1, 1, 4, 0, 128, 128, 0>"),
     ("b", 5, 64, 256, "gemm_dma_kernel<2, 4, 1, 1, 8, 0, 256, 256, 1>")],  # 256 rows of B
)
def test_i8_products_over_an_operand(cuda, how, operand, blocks, t, n, kernel):
    """Each Block's product stored over its own tile of A or B, as one memref of
    the program and as one tensor passed for both: the oracle's bytes of the
    product stored elsewhere."""
    import torch

    apart, over = i8_over(operand, blocks, t, n)
    rng = np.random.default_rng(n)
    shape = {"a": [(blocks * t, n), (n, n)], "b": [(n, n), (n, blocks * t)]}[operand]
    a, b = (rng.integers(-3, 4, s, dtype=np.int8) for s in shape)
    at = "ab".index(operand)
    want = run_oracle(apart, [a, b, np.zeros_like((a, b)[at])], oracle_threads())[2]
    dev = [to_device(x, "i8", cuda) for x in (a, b, np.zeros_like((a, b)[at]))]
    print(f"[gpu] i8 product over {operand}, {how}: {xt.plan(over)['kernel']}", flush=True)
    if how == "one memref":
        xt.launch(over, *dev)
    else:
        xt.launch(apart, dev[0], dev[1], dev[at])
    torch.cuda.synchronize()
    assert np.array_equal(dev[at].cpu().numpy(), want)
    assert kernels_of(*((over, dev) if how == "one memref" else (apart, [dev[0], dev[1], dev[at]]))) == [kernel]


def test_one_row_over_its_bias(cuda):
    """c = a @ b + c over one row, c of two column Blocks: the sum's own memref as
    the bias."""
    k, n, tn = 72, 180, 90
    m = xt.convert(_row_plus_kernel, args=(xt.Array((1, k), xt.float16), xt.Array((k, n), xt.float16),
                                          xt.Array((1, n), xt.float32), k, tn), grid=(2, 1, 1))
    assert " gemm k=72" in xt.plan(m)["kernel"]
    rng = np.random.default_rng(2)
    a, b = _narrow(rng, (1, k), "f16"), _narrow(rng, (k, n), "f16")
    c = rng.uniform(-1, 1, (1, n)).astype(np.float32)
    got = run_gpu(m, [a, b, c], ["f16", "f16", "f32"], cuda, case="one row over its bias")[2]
    assert frob_rel(got, closed_form.matmul(_wide(a), _wide(b)) + c) <= _bar(k)


@xt.kernel
def _row_plus_kernel(a, b, c, k, tn):
    j = xt.bid(0)
    x = xt.load(a, index=(0, 0), shape=(1, k), shared=1)
    w = xt.load(b, index=(0, j), shape=(k, tn))
    bias = xt.load(c, index=(0, j), shape=(1, tn))
    xt.store(c, index=(0, j), tile=xt.matmul(x, w) + bias)
