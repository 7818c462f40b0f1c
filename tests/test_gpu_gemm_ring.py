"""FP16 products and convolutions on four-wave tiles over a ring of LDS stages (MI355X_FP16/gemm_ring.hip): every configuration at the edges of its
tiles, through the C ABI."""
import numpy as np
import pytest
import torch

from utils.helix_runtime import load
from utils.hip_ctypes import HELIX_ERR_INVALID_VALUE, HELIX_ERR_UNSUPPORTED
from MI355X_FP16 import build_MI355X_FP16 as b16
from oracle import oracle as O
from gpu_helpers import dev, run_conv, run_gemm_f16

pytestmark = pytest.mark.gpu

# M, N, K, columns of padding behind the rows of A and B
PROBLEMS = [(1, 1, 8, 0),              # one row, one column, a K tile of one chunk
            (33, 47, 40, 8),           # N odd: results by halves
            (257, 130, 64, 0),         # one K tile; results two halves at a time
            (70, 300, 712, 16),        # a narrow first K tile; four halves at a time
            (225, 161, 200, 0),        # one beyond the largest tile's rows, fewer K tiles than stages and one
            (513, 520, 320, 0)]        # several tiles both ways, eight halves at a time


@pytest.mark.parametrize("problem", PROBLEMS, ids=lambda p: "x".join(map(str, p)))
def test_every_configuration_integer_exact(problem):
    M, N, K, pad = problem
    rng = np.random.default_rng(sum(problem))
    A = rng.integers(-2, 3, (M, K)).astype(np.float16)
    B = rng.integers(-1, 2, (K, N)).astype(np.float16)
    exact = A.astype(np.int64) @ B.astype(np.int64)
    assert np.abs(exact).max() < 2048
    for key in b16.RING_KEYS:
        got = run_gemm_f16(load(b16.library_for_key(key)), A, B, ldpad=pad)
        assert np.array_equal(got.astype(np.int64), exact), key


def test_many_tiles_integer_exact():
    """More tiles than the chip holds at once, many K tiles; the whole result against the exact product on the device."""
    M, N, K = 3000, 3080, 1000
    rng = np.random.default_rng(5)
    dA, dB = dev(rng.integers(-2, 3, (M, K)).astype(np.float16)), dev(rng.integers(-1, 2, (N, K)).astype(np.float16))
    want = (dA.float() @ dB.float().t())
    assert want.abs().max() < 2048
    for key in b16.RING_KEYS:
        C = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda:0")
        load(b16.library_for_key(key)).gemm(dA.data_ptr(), dB.data_ptr(), C.data_ptr(), M, N, K, K, K, N)
        assert torch.equal(C.float(), want), key


def test_results_stay_inside_their_rows():
    """ldc beyond N and a C off the vector alignment; neighbours keep what they held."""
    rng = np.random.default_rng(6)
    A = rng.integers(-2, 3, (100, 72)).astype(np.float16)
    B = rng.integers(-1, 2, (90, 72)).astype(np.float16)
    exact = (A.astype(np.int64) @ B.T.astype(np.int64)).astype(np.float32)
    dA, dB = dev(A), dev(B)
    for key in b16.RING_KEYS[::4]:
        for ldc, offset in ((96, 0), (92, 4), (94, 2), (93, 1)):
            out = torch.full((100 * ldc + 16,), 7.0, dtype=torch.float16, device="cuda:0")
            load(b16.library_for_key(key)).gemm(dA.data_ptr(), dB.data_ptr(), out.data_ptr() + 2 * offset, 100, 90, 72, 72, 72, ldc)
            got = out.cpu().numpy().astype(np.float32)
            rows = got[offset:offset + 100 * ldc].reshape(100, ldc)
            assert np.array_equal(rows[:, :90], exact), (key, ldc)
            assert (rows[:, 90:] == 7).all() and (got[:offset] == 7).all() and (got[offset + 100 * ldc:] == 7).all(), (key, ldc)


def test_infinities_stay_in_their_row_and_column():
    """K of one chunk beyond a tile: what the copies do not fetch is zero, not what LDS or the next row holds."""
    A = np.zeros((40, 72), np.float16)
    B = np.zeros((72, 50), np.float16)
    A[7, 71], B[71, 9] = np.inf, 1
    A[8, :], B[0, 9] = 1, 1
    want = np.zeros((40, 50), np.float32)
    want[7, :] = np.nan
    want[7, 9] = np.inf
    want[8, 9] = 2
    for key in b16.RING_KEYS[::3]:
        got = run_gemm_f16(load(b16.library_for_key(key)), A, B)
        assert np.array_equal(got.astype(np.float32), want, equal_nan=True), key


def test_graph_replays_and_refusals():
    rng = np.random.default_rng(8)
    A = rng.integers(-2, 3, (130, 200)).astype(np.float16)
    B = rng.integers(-1, 2, (200, 90)).astype(np.float16)
    exact = A.astype(np.int64) @ B.astype(np.int64)
    dA, dB = dev(A), dev(np.ascontiguousarray(B.T))
    lib = load(b16.library_for_key(b16.RING_KEYS[0]))
    C = torch.zeros((130, 90), dtype=torch.float16, device="cuda:0")
    args = (dA.data_ptr(), dB.data_ptr(), C.data_ptr(), 130, 90, 200, 200, 200, 90)
    lib.gemm(*args)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        lib.gemm(*args, 0, 0, torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        C.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(C.cpu().numpy().astype(np.int64), exact)
    assert lib.gemm(*args[:5], 199, *args[6:], check=False) == HELIX_ERR_INVALID_VALUE
    assert lib.gemm(dA.data_ptr() + 2, *args[1:], check=False) == HELIX_ERR_INVALID_VALUE
    conv = (dA.data_ptr(), dB.data_ptr(), C.data_ptr(), 1, 8, 8)
    assert lib.conv2d(*conv, 12, 8, 1, 1, 1, 0, check=False) == HELIX_ERR_UNSUPPORTED      # chunks across taps
    assert lib.conv2d(*conv, 8, 8, 4, 8, 1, 0, check=False) == HELIX_ERR_UNSUPPORTED       # 32 taps
    assert lib.conv2d(dA.data_ptr() + 2, *conv[1:], 8, 8, 3, 3, 1, 1, check=False) == HELIX_ERR_INVALID_VALUE
    x = rng.integers(-1, 2, (3, 5, 7, 72)).astype(np.float16)
    w = rng.integers(-1, 2, (40, 1, 1, 72)).astype(np.float16)
    want = O.conv2d_nhwc(x.astype(np.float32), w.astype(np.float32), 1, 0)
    for key in b16.RING_KEYS[::5]:
        assert np.array_equal(run_conv(load(b16.library_for_key(key)), x, w, 1, 0, torch.float16).astype(np.float32), want), key


# batch, channels, H, W, filters, kH, kW, stride, pad
LAYERS = [(1, 8, 3, 3, 1, 3, 3, 1, 0),         # one pixel, nine taps of a chunk in two tiles
          (2, 64, 9, 11, 70, 3, 3, 1, 1),      # a tile is one tap; filters two at a time
          (3, 24, 14, 10, 33, 5, 5, 2, 2),     # a tile over three taps
          (2, 128, 12, 12, 48, 5, 5, 1, 4),    # rows and columns of taps beyond the image
          (2, 104, 7, 7, 40, 1, 1, 2, 0),      # strided 1 x 1: no plain product
          (2, 8, 9, 12, 20, 5, 6, 1, 0),       # 30 taps, eight of them a tile
          (1, 16, 40, 3, 24, 31, 1, 3, 2),     # 31 taps
          (2, 192, 20, 23, 260, 3, 2, 3, 1)]   # several tiles both ways, rows off every multiple


@pytest.mark.parametrize("layer", LAYERS, ids=lambda l: "x".join(map(str, l)))
def test_every_configuration_convolves_integer_exact(layer):
    B, IC, H, W, OC, kH, kW, stride, pad = layer
    rng = np.random.default_rng(sum(layer))
    x = rng.integers(-1, 2, (B, H, W, IC)).astype(np.float16)
    w = rng.integers(-1, 2, (OC, kH, kW, IC)).astype(np.float16)
    want = O.conv2d_nhwc(x.astype(np.float32), w.astype(np.float32), stride, pad)
    assert np.abs(want).max() < 2048
    for key in b16.RING_KEYS:
        got = run_conv(load(b16.library_for_key(key)), x, w, stride, pad, torch.float16)
        assert np.array_equal(got.astype(np.float32), want), key


def test_infinities_in_the_input_reach_their_pixels_only():
    """Padding, channels beyond the last tile and rows beyond the last pixel are zeros, not what lies beside them."""
    x = np.zeros((2, 6, 7, 40), np.float16)
    w = np.ones((35, 3, 3, 40), np.float16)
    x[0, 5, 6, 39] = np.inf
    want = np.zeros((2, 6, 7, 35), np.float32)
    want[0, 4:6, 5:7] = np.inf
    for key in b16.RING_KEYS:
        got = run_conv(load(b16.library_for_key(key)), x, w, 1, 1, torch.float16)
        assert np.array_equal(got.astype(np.float32), want), key
