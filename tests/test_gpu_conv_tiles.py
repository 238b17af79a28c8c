"""GPU parity of the small-tile implicit GEMM (kernels/conv_tiles.hip) where its
tiles, stages and taps do not line up: pixels past the last tile, K ending inside
a stage, taps of three or five 16-byte chunks, windows outside the image, few and
many output channels; and of conv_igemm.hip on the same layers
(XTILE_AMD_CONV_IGEMM=1), which no longer takes them by itself.

f16 / bf16 against the oracle within 4 sqrt(K) 2^-24 (K f32 additions of random
sign, each rounding by at most 2^-24 of its partial sum); i8 exact."""

from __future__ import annotations

import numpy as np
import pytest

import xtile_amd as xt
from oracle import f32_to_bf16_bits
from tests.conftest import oracle_threads
from tests.gpu_util import frob_rel, run_gpu, run_oracle
from xtile_amd import kernels as K

pytestmark = pytest.mark.gpu

_XT = {"f16": xt.float16, "bf16": xt.bfloat16, "i8": xt.int8}


def _conv(cuda, n, h, w, cin, cout, kh, kw, pad, stride, dil, dt, kernels):
    oh = (h + pad[0] + pad[2] - dil[0] * (kh - 1) - 1) // stride[0] + 1
    ow = (w + pad[1] + pad[3] - dil[1] * (kw - 1) - 1) // stride[1] + 1
    mod = K.conv2d(n, h, w, cin, cout, kh, kw, 1, ow, dtype=_XT[dt], pad=pad, stride=stride, dilation=dil)
    rng = np.random.default_rng(h * cin)
    if dt == "i8":
        x = rng.integers(-128, 128, (n, h, w, cin), dtype=np.int8)
        f = rng.integers(-128, 128, (kh, kw, cin, cout), dtype=np.int8)
    else:
        x = rng.normal(0, 0.1, (n, h, w, cin)).astype(np.float32)
        f = rng.normal(0, 0.1, (kh, kw, cin, cout)).astype(np.float32)
        x, f = (x.astype(np.float16), f.astype(np.float16)) if dt == "f16" else (f32_to_bf16_bits(x), f32_to_bf16_bits(f))
    bufs = [x, f, np.full((n, oh, ow, cout), np.nan, np.float32)]
    got = run_gpu(mod, bufs, [dt, dt, "f32"], cuda, case=f"conv {kernels[-1]} {n}x{h}x{w}x{cin}->{cout} {kh}x{kw} {dt}",
                  kernels=kernels)[2]
    want = run_oracle(mod, bufs, oracle_threads())[2]
    if dt == "i8":
        assert np.array_equal(got, want)
    else:
        assert frob_rel(got, want) <= 4 * np.sqrt(kh * kw * cin) * 2.0**-24


_ELEM = {"f16": 0, "bf16": 1, "i8": 2}


def _tiles(dt, bm, bn, part=0):
    return [f"conv_tiles_kernel<{_ELEM[dt]}, {bm}, {bn}, {part}>"]


def _igemm(dt, bm, bn, part=0, split=False):
    """128-row tiles with loader waves, 256 x 64 without."""
    rest = "64, 64, 64, 0" if bm == 256 else f"64, {bn // 2}, 128, 8"
    return ["ig_zero_kernel"] * split + [f"conv_igemm_kernel<{_ELEM[dt]}, {bm}, {bn}, {rest}, {part}, 4>"]


def _deep(dt, split=False):
    return ["ig_zero_kernel"] * split + [f"conv_igemm_kernel<{_ELEM[dt]}, 64, 128, 32, 64, 128, 8, 0, 4>"]


# (layer), the kernel of its own choice, the one with XTILE_AMD_CONV_IGEMM=1
_LAYERS = [
    ((1, 1, 1, 512, 8, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1), "f16"),        # one pixel, one stage of 8 channels
     _tiles("f16", 32, 32), _igemm("f16", 128, 64)),
    ((1, 5, 7, 264, 40, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "bf16"),      # taps of 33 chunks
     _tiles("bf16", 32, 32), _igemm("bf16", 256, 64, split=True)),
    ((3, 9, 9, 24, 200, 5, 5, (2, 2, 2, 2), (1, 1), (1, 1), "f16"),       # taps of 3 chunks, channels past 192
     _tiles("f16", 32, 32), _igemm("f16", 128, 64)),
    ((2, 13, 11, 40, 256, 5, 3, (0, 1, 3, 2), (2, 1), (1, 2), "bf16"),    # taps of 5, uneven pads, strides, dilations
     _tiles("bf16", 32, 32), _igemm("bf16", 128, 64)),
    ((1, 33, 31, 136, 72, 3, 3, (1, 1, 1, 1), (2, 2), (2, 2), "f16"),     # windows half outside
     _tiles("f16", 32, 32), _igemm("f16", 128, 64)),
    ((1, 20, 20, 48, 48, 7, 7, (3, 3, 3, 3), (1, 1), (1, 1), "i8"),       # taps of 3 chunks of bytes
     _tiles("i8", 32, 32), _igemm("i8", 128, 64)),
    ((5, 18, 18, 512, 32, 3, 3, (1, 1, 1, 1), (2, 2), (1, 1), "i8"),
     _tiles("i8", 32, 32), _igemm("i8", 128, 64)),
    ((2, 7, 7, 96, 528, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1), "i8"),
     _tiles("i8", 32, 32), _igemm("i8", 128, 128)),
    ((9, 23, 23, 48, 64, 5, 5, (2, 2, 2, 2), (1, 1), (1, 1), "f16"),
     _tiles("f16", 32, 64), _igemm("f16", 128, 64)),
    ((1, 1, 1, 20, 16, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1), "i8"),         # a last chunk of 4 channels of its own
     _tiles("i8", 32, 32, 1), _igemm("i8", 128, 128, 1)),
    ((1, 9, 7, 44, 32, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "i8"),         # of 12
     _tiles("i8", 32, 32, 1), _igemm("i8", 128, 64, 1)),
    ((2, 13, 11, 40, 272, 5, 3, (0, 1, 3, 2), (2, 1), (1, 2), "i8"),      # of 8, uneven pads, strides, dilations
     _tiles("i8", 32, 32, 1), _igemm("i8", 128, 64, 1)),
    ((3, 19, 19, 500, 64, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "i8"),      # of 4 after several stages
     _tiles("i8", 32, 32, 1), _igemm("i8", 128, 64, 1)),
    ((9, 23, 23, 28, 64, 5, 5, (2, 2, 2, 2), (1, 1), (1, 1), "i8"),
     _tiles("i8", 32, 64, 1), _igemm("i8", 128, 64, 1)),
    ((19, 112, 112, 20, 16, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "i8"),
     ["conv2d_small_kernel<2, 0, 0, 0>"], _igemm("i8", 256, 64, 1)),
    ((2, 11, 11, 512, 512, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "f16"),    # 64 x 128 tiles, their K split
     _deep("f16", split=True), None),
    ((20, 17, 17, 256, 256, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "i8"),    # whole
     _deep("i8"), None),
    ((50, 40, 40, 96, 64, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "bf16"),    # bands of four rows, half the filter's bytes
     ["conv2d_band_kernel<2, 6, 1>"], None),
    ((53, 21, 21, 64, 128, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "f16"),    # of two rows, a tenth of them
     _igemm("f16", 128, 128), None),
    ((2, 65, 65, 16, 128, 1, 1, (0, 0, 0, 0), (2, 2), (1, 1), "bf16"),
     _tiles("bf16", 32, 64), None),
    ((7, 24, 24, 16, 96, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1), "i8"),
     _tiles("i8", 32, 64), None),
    ((4, 23, 23, 16, 256, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "f16"),
     _tiles("f16", 64, 64), None),
    ((3, 54, 54, 16, 56, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "bf16"),     # a channel tile of 56
     _tiles("bf16", 64, 64), None),
    ((22, 10, 10, 16, 256, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "i8"),
     _tiles("i8", 64, 64), None),
    ((2, 25, 25, 40, 512, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1), "i8"),
     _tiles("i8", 64, 64, 1), None),
]


@pytest.mark.parametrize("layer,kernels,forced", [(x, own, False) for x, own, _ in _LAYERS] +
                         [(x, igemm, True) for x, _, igemm in _LAYERS if igemm])
def test_conv_tiles(cuda, monkeypatch, layer, kernels, forced):
    monkeypatch.setenv("XTILE_AMD_CONV_IMAGE", "0")
    if forced:
        monkeypatch.setenv("XTILE_AMD_CONV_IGEMM", "1")
    _conv(cuda, *layer, kernels)


@pytest.mark.parametrize(
    "n,h,cin,cout,k,pad,stride,dt,kernels",
    [(20, 28, 128, 128, 3, 1, 1, "f16", _deep("f16")),                # two stages a tap
     (32, 28, 128, 128, 3, 1, 1, "f16", _igemm("f16", 128, 128)),
     (17, 37, 136, 96, 3, 1, 1, "bf16", _igemm("bf16", 128, 128)),    # channels past Cout, stages past a tap's channels
     (13, 47, 96, 64, 5, 2, 2, "f16", _igemm("f16", 256, 64, split=True)),  # pixels past the last tile
     (53, 47, 40, 64, 5, 2, 2, "bf16", _igemm("bf16", 128, 64)),      # pixels past the last tile
     (32, 28, 128, 128, 3, 1, 1, "i8", _igemm("i8", 128, 128)),       # i8 whose filter leaves bands of one row
     (26, 28, 192, 80, 5, 2, 1, "i8", _igemm("i8", 128, 128)),        # channels past Cout
     (26, 28, 172, 80, 5, 2, 1, "i8", _igemm("i8", 128, 128, 1)),     # the same, the last chunk of a tap 12 channels
     (32, 28, 132, 128, 3, 1, 1, "i8", _igemm("i8", 128, 128, 1))],   # of 4 channels
)
def test_conv_loader_waves(cuda, monkeypatch, n, h, cin, cout, k, pad, stride, dt, kernels):
    """conv_igemm.hip's 128 x 128 and 128 x 64 tiles with loader waves, and the 64 x
    128 tiles and the split that two of the layers take instead."""
    monkeypatch.setenv("XTILE_AMD_CONV_IGEMM", "1")
    _conv(cuda, n, h, h, cin, cout, k, k, (pad,) * 4, (stride, stride), (1, 1), dt, kernels)
