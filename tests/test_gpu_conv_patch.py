"""Convolutions whose input stays in LDS (common/helix_conv_patch.h), FP16 and FP32: every configuration on layers at the edges
of its blocks, through the C ABI."""
import numpy as np
import pytest
import torch

from utils.helix_runtime import load
from utils.hip_ctypes import HELIX_ERR_INVALID_VALUE, HELIX_ERR_UNSUPPORTED
from MI355X_FP16 import build_MI355X_FP16 as b16
from MI355X_FP16 import MI355X_FP16_conv as c16
from MI355X_FP32 import build_MI355X_FP32 as b32
from MI355X_FP32 import MI355X_FP32_conv as c32
from oracle import oracle as O
from gpu_helpers import conv_out_hw, dev, run_conv

pytestmark = pytest.mark.gpu

# (batch, IC, H, W, OC, kH, kW, stride, pad)
LAYERS = [(1, 8, 1, 1, 1, 1, 1, 1, 0),            # one pixel, one channel, K of one chunk
          (3, 8, 5, 7, 3, 3, 3, 1, 1),            # K of nine chunks, several images in a block, channels off the vector width
          (2, 24, 9, 11, 20, 3, 3, 2, 1),         # an odd number of chunks per pixel, stride 2
          (5, 16, 3, 2, 33, 2, 2, 1, 2),          # padding wider than the image's edge
          (2, 40, 13, 6, 64, 1, 5, 3, 0),         # stride beyond the filter's height
          (1, 64, 17, 19, 130, 3, 3, 1, 1),       # whole K tiles, ragged blocks both ways
          (7, 32, 7, 7, 48, 5, 5, 1, 2),          # images across blocks
          (9, 72, 4, 33, 16, 1, 1, 1, 0),         # pointwise
          (1, 8, 60, 120, 8, 7, 3, 4, 3)]         # more staged pixels than a thread's batch of loads


# channel counts off the chunk: FP32 only
LAYERS32 = LAYERS + [(2, 3, 21, 23, 40, 7, 7, 2, 3),     # one chunk per pixel, three floats of it
                     (1, 1, 9, 17, 5, 3, 3, 1, 1),
                     (3, 25, 10, 9, 17, 3, 3, 1, 1),     # a last chunk of one float; channels off the store's width
                     (2, 6, 8, 8, 36, 1, 3, 1, 0),
                     (1, 7, 1, 3, 16, 1, 1, 1, 0)]
CASES = [(np.float16, b16, c16, l) for l in LAYERS] + [(np.float32, b32, c32, l) for l in LAYERS32]


@pytest.mark.parametrize("dtype,build,conv,layer", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else getattr(v, "__name__", "").split(".")[-1])
def test_every_configuration_integer_exact(dtype, build, conv, layer):
    """Inputs in {-1, 0, 1}: exact in any order of the sums."""
    batch, IC, H, W, OC, kH, kW, stride, pad = layer
    rng = np.random.default_rng(sum(layer))
    x = rng.integers(-1, 2, (batch, H, W, IC)).astype(dtype)
    w = rng.integers(-1, 2, (OC, kH, kW, IC)).astype(dtype)
    want = O.conv2d_nhwc(x.astype(np.float32), w.astype(np.float32), stride, pad)
    assert np.abs(want).max() < 2048
    ran = 0
    for point in build.PATCH_POINTS:
        if conv.PATCH.layout(point, *layer) is None:
            continue
        got = run_conv(load(build.library_for_key(build.patch_key(point))), x, w, stride, pad, torch.float16 if dtype is np.float16 else torch.float32)
        assert np.array_equal(got.astype(np.float32), want), point
        ran += 1
    assert ran >= 4


@pytest.mark.parametrize("IC", [8, 3])
@pytest.mark.parametrize("dtype,build", [(np.float16, b16), (np.float32, b32)])
def test_infinite_pixel_reaches_its_window_only(dtype, build, IC):
    """K has a remainder, which multiplies zeros by zeros, whatever lies beside them; so have the channels with IC = 3."""
    if dtype is np.float16 and IC % 8:
        pytest.skip("whole chunks only")
    x = np.zeros((2, 12, 16, IC), dtype)
    x[1, 6, 8, IC - 1] = np.inf
    x[1, 11, 15, 0] = np.nan
    w = np.ones((40, 3, 3, IC), dtype)
    want = np.zeros((2, 12, 16, 1), dtype)
    want[1, 5:8, 7:10] = np.inf
    want[1, 10:, 14:] = np.nan
    for key in build.patch_keys()[::3]:
        got = run_conv(load(build.library_for_key(key)), x, w, 1, 1, torch.float16 if dtype is np.float16 else torch.float32)
        assert np.array_equal(got, np.repeat(want, 40, axis=3), equal_nan=True), key


def test_infinite_weight_of_the_next_tap():
    """FP32, three channels: the fourth float of a tap's chunk would be the next tap's first."""
    x = np.zeros((1, 5, 5, 3), np.float32)
    x[0, 2, 2] = 1
    w = np.zeros((16, 3, 3, 3), np.float32)
    w[:, 1, 1, 0] = np.inf
    for key in b32.patch_keys()[::3]:
        got = run_conv(load(b32.library_for_key(key)), x, w, 1, 1, torch.float32)
        # zero times the infinite weight is NaN at every other pixel; with the zero behind the chunk before it, it is not one here
        assert np.isposinf(got[0, 2, 2]).all() and np.isnan(got).sum() == 24 * 16, key


@pytest.mark.parametrize("offset", [1, 4])
def test_results_off_the_vector_alignment(offset):
    """A y that is not aligned to a lane's store is written by halves; x and w off 16 bytes are refused, as elsewhere."""
    rng = np.random.default_rng(offset)
    x = rng.integers(-1, 2, (2, 9, 9, 16)).astype(np.float16)
    w = rng.integers(-1, 2, (64, 3, 3, 16)).astype(np.float16)
    want = O.conv2d_nhwc(x.astype(np.float32), w.astype(np.float32), 1, 1)
    dx, dw = dev(x), dev(w)
    for key in b16.patch_keys()[::7]:
        lib = load(b16.library_for_key(key))
        out = torch.full((want.size + 16,), 7.0, dtype=torch.float16, device="cuda:0")
        lib.conv2d(dx.data_ptr(), dw.data_ptr(), out.data_ptr() + 2 * offset, 2, 9, 9, 16, 64, 3, 3, 1, 1)
        got = out.cpu().numpy().astype(np.float32)
        assert np.array_equal(got[offset:offset + want.size], want.ravel()), key
        assert (got[:offset] == 7).all() and (got[offset + want.size:] == 7).all(), key
        assert lib.conv2d(dx.data_ptr() + 2, dw.data_ptr(), out.data_ptr(), 1, 8, 8, 16, 64, 3, 3, 1, 1, check=False) == HELIX_ERR_INVALID_VALUE
        assert lib.conv2d(dx.data_ptr(), dw.data_ptr(), out.data_ptr(), 1, 8, 8, 12, 8, 3, 3, 1, 1, check=False) == HELIX_ERR_UNSUPPORTED
        assert lib.gemm(dx.data_ptr(), dw.data_ptr(), out.data_ptr(), 16, 16, 16, 16, 16, 16, check=False) == HELIX_ERR_UNSUPPORTED
