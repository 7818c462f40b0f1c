"""FP16 convolutions of one to four input channels (common/helix_conv_thin.h) through the C ABI: filters of every
kernel variant (2, 4 and 7 MFMA steps of weights in registers, longer ones in LDS), both stride parities, blocks with
ragged edges, rows cut into column blocks, several blocks per workgroup, output channels off the vector and tile widths."""
import numpy as np
import pytest
import torch

from utils.helix_runtime import load
from MI355X_FP16 import build_MI355X_FP16 as b16
from oracle import oracle as O
from gpu_helpers import run_conv

pytestmark = pytest.mark.gpu

# (batch, IC, H, W, OC, kH, kW, stride, pad)
LAYERS = [(1, 3, 1, 8, 1, 1, 1, 1, 0),            # one row, one output channel
          (1, 3, 2, 3, 8, 1, 1, 1, 0),            # fewer pixels than a staging unit's window
          (2, 3, 17, 16, 64, 3, 3, 1, 1),         # 2 steps, odd stride
          (3, 3, 33, 31, 72, 3, 3, 2, 1),         # odd width and an odd number of halves in x; a second channel block
          (1, 3, 90, 101, 16, 3, 5, 3, 4),        # filter wider than high, padding beyond the filter's half
          (2, 3, 24, 25, 65, 5, 5, 1, 2),         # 4 steps, one channel in the second block
          (2, 3, 40, 44, 64, 7, 7, 2, 3),         # 7 steps
          (1, 3, 30, 170, 24, 7, 7, 1, 3),        # ... with rows cut into column blocks
          (130, 3, 30, 29, 96, 11, 11, 4, 0),     # weights in LDS, several blocks per workgroup
          (1, 1, 40, 300, 32, 5, 20, 2, 0),       # one channel, a long filter: too few pixels, takes the column buffer
          (2, 2, 9, 11, 12, 7, 6, 1, 5),          # two channels, even filter width, padding wider than the image's edge
          (1, 4, 30, 31, 70, 3, 3, 1, 1),
          (600, 3, 20, 20, 8, 3, 3, 1, 1)]        # more blocks than the chip holds at once


@pytest.mark.parametrize("layer", LAYERS, ids=lambda l: "x".join(map(str, l)))
def test_thin_convolution_integer_exact(layer):
    """Inputs in {-1, 0, 1}: every product and partial sum is a small integer, so the result is exact in any order."""
    batch, IC, H, W, OC, kH, kW, stride, pad = layer
    rng = np.random.default_rng(sum(layer))
    x = rng.integers(-1, 2, (batch, H, W, IC)).astype(np.float16)
    w = rng.integers(-1, 2, (OC, kH, kW, IC)).astype(np.float16)
    want = O.conv2d_nhwc(x.astype(np.float32), w.astype(np.float32), stride, pad)
    assert np.abs(want).max() < 2048
    got = run_conv(load(b16.kernel_library("gemm", 2, 64, 64, 32, 32, 64)), x, w, stride, pad, torch.float16)
    assert np.array_equal(got.astype(np.float32), want)


@pytest.mark.parametrize("kW", [3, 5, 7])
def test_thin_convolution_reads_only_the_filter_window(kW):
    """An infinite pixel reaches exactly the outputs whose window holds it: the second pixel of a pair that hangs over
    the end of a filter row does not count."""
    x = np.zeros((1, 12, 16, 3), np.float16)
    x[0, 6, 8, 1] = np.inf
    w = np.ones((8, kW, kW, 3), np.float16)
    got = run_conv(load(b16.kernel_library("gemm", 2, 64, 64, 32, 32, 64)), x, w, 1, kW // 2, torch.float16)
    want = np.zeros((12, 16), bool)
    h = kW // 2
    want[max(0, 6 - h):6 + h + 1, max(0, 8 - h):8 + h + 1] = True
    assert np.array_equal(np.isinf(got[0]), np.repeat(want[:, :, None], 8, axis=2))
    assert np.array_equal(got[0][~want], np.zeros_like(got[0][~want]))


@pytest.mark.parametrize("layer", [(1, 3, 9, 171, 24, 7, 7, 1, 3), (5, 3, 7, 7, 8, 3, 3, 1, 1), (1, 3, 31, 31, 64, 11, 11, 4, 2),
                                   (301, 3, 5, 9, 16, 5, 5, 1, 2), (1, 3, 3, 5, 8, 2, 2, 1, 1)], ids=lambda l: "x".join(map(str, l)))
def test_last_half_of_an_odd_input(layer):
    """An odd number of halves: the last one lies in no whole dword and is read by itself, in every block whose patch holds
    its pixel (several rows of blocks, column blocks, weights in registers and in LDS)."""
    batch, IC, H, W, OC, kH, kW, stride, pad = layer
    assert batch * IC * H * W % 2 == 1
    x = np.zeros((batch, H, W, IC), np.float16)
    x[-1, -1, -1, :] = 1, 2, 4
    w = np.random.default_rng(7).integers(1, 4, (OC, kH, kW, IC)).astype(np.float16)
    want = O.conv2d_nhwc(x.astype(np.float32), w.astype(np.float32), stride, pad)
    assert want.max() > 0
    got = run_conv(load(b16.kernel_library("gemm", 2, 64, 64, 32, 32, 64)), x, w, stride, pad, torch.float16)
    assert np.array_equal(got.astype(np.float32), want)


@pytest.mark.parametrize("layer", [(3, 3, 210, 211, 72, 3, 3, 1, 1), (2, 3, 257, 257, 96, 5, 5, 1, 2), (9, 3, 242, 243, 65, 4, 4, 2, 2),
                                   (3, 3, 210, 208, 97, 3, 3, 1, 1)], ids=lambda l: "x".join(map(str, l)))
def test_many_pixels_of_up_to_96_channels(layer):
    """96 channels per workgroup from 131072 pixels on (2 and 4 steps), the edges of its channel range and one beyond it."""
    test_thin_convolution_integer_exact(layer)
