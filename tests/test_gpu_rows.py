"""GPU parity of the flat elementwise kernel and the row softmax where rows and
runs are not whole vectors, waves or workgroups, and in buffers off the vector
alignment.  Bars: add bit-exact; softmax 1e-5 relative to its float64 closed form
(absolute below FLT_MIN)."""

from __future__ import annotations

import numpy as np
import pytest

import xtile_amd as xt
from oracle import closed_form
from tests.gpu_util import kernels_of
from xtile_amd import kernels as K

pytestmark = pytest.mark.gpu


def _views(cuda, off, *arrays):
    """The arrays on the GPU, each `off` elements past an aligned address, with
    guard elements around them."""
    import torch

    flats, views = [], []
    for x in arrays:
        flat = torch.full((x.size + off + 8,), 7.0, device=cuda)
        flat[off : off + x.size] = torch.from_numpy(x).reshape(-1).to(cuda)
        flats.append(flat)
        views.append(flat[off : off + x.size].view(x.shape))
    return flats, views


def _run(cuda, m, off, case, *arrays):
    import torch

    flats, views = _views(cuda, off, *arrays)
    print(f"[gpu] {case} {off} elements off: {xt.plan(m)['kernel']}", flush=True)
    xt.launch(m, *views)
    torch.cuda.synchronize()
    out = flats[-1].cpu().numpy()
    assert np.all(out[:off] == 7.0) and np.all(out[off + arrays[-1].size :] == 7.0)
    return views[-1].cpu().numpy()


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("rows,cols,tm,tn", [(1, 3, 1, 3), (2, 2, 1, 2), (1, 5, 1, 1), (3, 683, 3, 683), (2, 1023, 1, 341),
                                             (64, 33, 16, 11), (41, 51, 41, 17)])
def test_flat_add(cuda, rows, cols, tm, tn, off):
    rng = np.random.default_rng(rows * cols)
    a, b = (rng.uniform(-1, 1, (rows, cols)).astype(np.float32) for _ in range(2))
    got = _run(cuda, K.add(rows, cols, tm, tn), off, f"add {rows}x{cols}", a, b, np.zeros_like(a))
    assert np.array_equal(got.view(np.uint32), (a + b).view(np.uint32))


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("rows,cols,trow", [(5, 1, 5), (6, 3, 2), (7, 4, 1), (130, 5, 10), (33, 8, 11), (9, 9, 3), (12, 63, 4),
                                            (10, 256, 2), (10, 257, 5), (4098, 100, 2), (4098, 130, 3), (14, 1023, 7),
                                            (6, 2047, 3), (8, 2048, 4), (6, 2052, 2), (5, 8188, 5), (6, 4096, 3)])
def test_row_softmax(cuda, rows, cols, trow, off):
    rng = np.random.default_rng(rows + cols)
    x = rng.normal(0, 2, (rows, cols)).astype(np.float32)
    got = _run(cuda, K.softmax(rows, cols, trow), off, f"softmax {rows}x{cols}/{trow}", x, np.zeros_like(x))
    np.testing.assert_allclose(got, closed_form.softmax_rows(x), rtol=1e-5, atol=1.2e-38)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("rows,cols,trow,groups", [(512, 1025, 1, "2, 256"), (513, 1025, 1, "5, 64"), (514, 1536, 2, "6, 64"),
                                                  (520, 1790, 4, "7, 64"), (516, 2047, 3, "8, 64"), (512, 2047, 4, "2, 256"),
                                                  (513, 1024, 1, "4, 64"), (5, 1024, 1, "4, 64")])
def test_few_long_rows(cuda, rows, cols, trow, groups, off):
    """Up to 512 rows of 1025 to 2048 floats take the workgroup, more a wave."""
    rng = np.random.default_rng(rows + cols)
    x = rng.normal(0, 2, (rows, cols)).astype(np.float32)
    m = K.softmax(rows, cols, trow)
    got = _run(cuda, m, off, f"softmax {rows}x{cols}/{trow}", x, np.zeros_like(x))
    np.testing.assert_allclose(got, closed_form.softmax_rows(x), rtol=1e-5, atol=1.2e-38)
    assert kernels_of(m, _views(cuda, off, x, np.zeros_like(x))[1]) == [f"row_softmax_kernel<{groups}, 0>"]


@pytest.mark.parametrize("rows,cols,trow,kernel", [((1 << 32) + 4096, 2, 4096, "row_softmax_kernel<1, 1, 1>"),
                                                  (8388611, 2048, 7, "row_softmax_wide_kernel<512, 1, 1>")])
def test_row_softmax_of_more_rows_than_a_launch_takes(cuda, rows, cols, trow, kernel):
    """More rows than 2^31 indices or one launch's 2^32 threads: the workgroups
    walk them.  In place (34 and 69 GB); row r's odd columns stand r % 1021 / 256
    above a row of its even ones, so a row written elsewhere shows."""
    import torch

    if torch.cuda.mem_get_info()[0] < rows * cols * 4 + (8 << 30):
        pytest.skip("not enough free memory on the GPU")
    base = torch.linspace(-1, 1, cols, device=cuda)
    chunk = (1 << 28) // cols

    def part(r0):
        step = (torch.arange(r0, min(r0 + chunk, rows), device=cuda) % 1021).float() / 256
        return base + step[:, None] * (torch.arange(cols, device=cuda) % 2)

    x = torch.empty(rows, cols, device=cuda)
    for r0 in range(0, rows, chunk):
        x[r0 : r0 + chunk] = part(r0)
    m = K.softmax(rows, cols, trow)
    print(f"[gpu] softmax of {rows} rows", flush=True)
    xt.launch(m, x, x)
    for r0 in range(0, rows, chunk):
        torch.testing.assert_close(x[r0 : r0 + chunk], torch.softmax(part(r0), dim=1), rtol=1e-5, atol=0)
    assert kernels_of(m, [x, x]) == [kernel]
    del x
    torch.cuda.empty_cache()
