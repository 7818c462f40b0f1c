"""FP32 products and convolutions on four-wave tiles over a ring of LDS stages (MI355X_FP32/gemm_ring.hip): every configuration at the edges of its
tiles, through the C ABI."""
import numpy as np
import pytest
import torch

from utils.helix_runtime import load
from utils.hip_ctypes import HELIX_ERR_INVALID_VALUE, HELIX_ERR_UNSUPPORTED
from MI355X_FP32 import build_MI355X_FP32 as b32
from MI355X_FP32 import MI355X_FP32_conv as c32
from oracle import oracle as O
from gpu_helpers import conv_out_hw, dev, run_conv, run_gemv_f32, run_sgemm_f32

pytestmark = pytest.mark.gpu

# M, N, K: one chunk; half a K tile and one beyond it, a whole one and one beyond; fewer K tiles than stages; one beyond the
# largest tiles' rows and columns; several tiles both ways
PROBLEMS = [(1, 1, 1), (33, 47, 16), (65, 130, 17), (70, 300, 32), (225, 161, 33), (130, 257, 100), (513, 520, 336)]


@pytest.mark.parametrize("problem", PROBLEMS, ids=lambda p: "x".join(map(str, p)))
def test_every_configuration_integer_exact(problem):
    M, N, K = problem
    rng = np.random.default_rng(sum(problem))
    A = rng.integers(-8, 9, (M, K)).astype(np.float32)
    B = rng.integers(-8, 9, (K, N)).astype(np.float32)
    exact = A.astype(np.int64) @ B.astype(np.int64)
    for key in b32.RING_KEYS:
        got = run_sgemm_f32(load(b32.library_for_key(key)), A, B)
        assert np.array_equal(got.astype(np.int64), exact), key


def test_sums_next_to_sgemm():
    """Results beyond 5 x 2^20: up to 256 of K their products are added in ascending k, each rounded, as in an unpartitioned launch of
    sgemm.hip; longer chains are cut there, half a K tile behind them included (the error of one product behind 256 is that of 257).  That leaves
    less error than its two K groups."""
    rng = np.random.default_rng(4)
    A, B = rng.standard_normal((2600, 272)).astype(np.float32), rng.standard_normal((272, 2500)).astype(np.float32)
    for K in (255, 256, 257, 272):
        plain = run_sgemm_f32(load(b32.default_library()), A[:, :K], B[:K], workspace=False)
        exact = A[:, :K].astype(np.float64) @ B[:K].astype(np.float64)
        for key in b32.RING_KEYS:
            got = run_sgemm_f32(load(b32.library_for_key(key)), A[:, :K], B[:K])
            assert np.array_equal(got, plain) if K <= 256 else error(got, exact) <= 1.01 * error(plain, exact), (key, K)
    A, B = rng.standard_normal((290, 2600)).astype(np.float32), rng.standard_normal((2600, 301)).astype(np.float32)
    exact = A.astype(np.float64) @ B.astype(np.float64)
    limit = error(run_sgemm_f32(load(b32.sgemm_library(64, 64, 32, 32, 32, 2)), A, B, workspace=False), exact)
    for key in b32.RING_KEYS:
        assert error(run_sgemm_f32(load(b32.library_for_key(key)), A, B), exact) <= limit, key


def error(got, exact):
    return np.linalg.norm(got - exact) / np.linalg.norm(exact)


# The norm of n results' errors scatters by sqrt(1 / 2 n) of itself between two ways of summing that are equally exact: four times that
def scatter(n):
    return 1 + 4 * (0.5 / n) ** 0.5


def wave_tiles(key):
    """16 x 16 tiles of a wave."""
    return (key[3] // 16) * (key[4] // 16)


@pytest.mark.parametrize("K", [200, 256, 257, 272, 480, 800])
def test_few_results_are_as_exact_as_k_groups(K):
    """Where sgemm.hip's fastest configurations have four or eight K groups; K = 257 and 272 end half a K tile behind a whole one."""
    rng = np.random.default_rng(K)
    A, B = rng.standard_normal((290, K)).astype(np.float32), rng.standard_normal((K, 301)).astype(np.float32)
    exact = A.astype(np.float64) @ B.astype(np.float64)
    limit = min(error(run_sgemm_f32(load(b32.sgemm_library(*c)), A, B, workspace=False), exact)
                for c in b32.iter_kgroup_configs() if c[5] in (4, 8))
    for key in b32.RING_KEYS:
        assert error(run_sgemm_f32(load(b32.library_for_key(key)), A, B), exact) <= limit * scatter(290 * 301), key


@pytest.mark.parametrize("K", [260, 500, 1400])
def test_few_columns_are_as_exact_as_the_gemv(K):
    rng = np.random.default_rng(K)
    A, B = rng.standard_normal((3000, K)).astype(np.float32), rng.standard_normal((K, 7)).astype(np.float32)
    exact = A.astype(np.float64) @ B.astype(np.float64)
    limit = error(run_gemv_f32(load(b32.kernel_library("gemv_fp32")), B.T, A.T).T, exact)
    for key in b32.RING_KEYS:
        if wave_tiles(key) <= 4:                         # what such problems are run on
            assert error(run_sgemm_f32(load(b32.library_for_key(key)), A, B), exact) <= limit * scatter(3000 * 7), key


def infinite_sums(A, B):
    """Products of positive operands whose rows 5, 9, 11 and 13 of the first end in inf, -inf, NaN and beyond the largest float."""
    K = A.shape[1]
    for k in (3, K // 2, K - 1):            # first, a middle and the last K tile, chains of different places in it
        A[5, k], A[9, k] = np.inf, -np.inf
    A[11, 20], A[11, 40] = np.inf, -np.inf
    A[13, 8:200:16] = 3e38
    with np.errstate(all="ignore"):
        want = (A.astype(np.float64) @ B.astype(np.float64)).astype(np.float32)
    assert np.isinf(want).sum() == 3 * B.shape[1] and np.isnan(want).sum() == B.shape[1]
    return want


@pytest.mark.parametrize("K", [256, 500, 1400])
@pytest.mark.parametrize("few_rows", [False, True])
def test_infinite_sums_of_few_rows_or_columns(few_rows, K):
    """What a compensated sum lacks has no value once the sum is infinite: it stays so, and is NaN only where products of both signs are."""
    rng = np.random.default_rng(K)
    A, B = rng.integers(1, 9, (300, K)).astype(np.float32), rng.integers(1, 9, (K, 7)).astype(np.float32)
    want = infinite_sums(A, B)
    for key in b32.RING_KEYS:
        lib = load(b32.library_for_key(key))
        got = run_sgemm_f32(lib, B.T, A.T).T if few_rows else run_sgemm_f32(lib, A, B)
        assert np.array_equal(got, want, equal_nan=True), key


@pytest.mark.parametrize("IC", [32, 36, 29])
def test_infinite_sums_of_few_channels(IC):
    """The same in convolutions, the ring tiles' (IC a multiple of 4) and those whose input stays in LDS; the finite results are exact."""
    rng = np.random.default_rng(IC)
    x, w = rng.integers(0, 3, (2, 10, 11, IC)).astype(np.float32), rng.integers(1, 4, (13, 3, 3, IC)).astype(np.float32)
    want = O.conv2d_nhwc(x, w, 1, 1)
    x[0, 3, 4, IC - 1], want[0, 2:5, 3:6] = np.inf, np.inf
    x[1, 9, 10, 0], want[1, 8:, 9:] = -np.inf, -np.inf
    x[1, 0, 0, 7], want[1, :2, :2] = np.nan, np.nan
    for key in (b32.RING_KEYS if IC % 4 == 0 else ()) + b32.patch_keys():
        if b32.is_patch_key(key) and c32.PATCH.layout((key[0], key[1], key[3], key[4], key[6]), 2, IC, 10, 11, 13, 3, 3, 1, 1) is None:
            continue
        assert np.array_equal(run_conv(load(b32.library_for_key(key)), x, w, 1, 1, torch.float32), want, equal_nan=True), key


def test_many_tiles_integer_exact():
    """More workgroups than the chip holds at once, many K tiles; the whole result against the product in 64 bits on the device."""
    M, N, K = 3000, 3080, 500
    rng = np.random.default_rng(5)
    dA, dB = dev(rng.integers(-8, 9, (K, M)).astype(np.float32)), dev(rng.integers(-8, 9, (K, N)).astype(np.float32))
    want = (dA.double().t().contiguous() @ dB.double()).float()
    for key in b32.RING_KEYS:
        C = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda:0")
        load(b32.library_for_key(key)).gemm(dA.data_ptr(), dB.data_ptr(), C.data_ptr(), M, N, K, M, N, N)
        assert torch.equal(C, want), key


def test_operand_beyond_2_gib_integer_exact():
    """A of 2.4 GB: what a copy has not got (columns beyond M and N, pieces that a wave has not) reads zeros behind a tile's rows, not
    data of the operand."""
    M, N, K = 1800003, 20, 331
    gen = torch.Generator(device="cuda:0").manual_seed(9)
    dA = torch.randint(-8, 9, (K, M + 1), generator=gen, device="cuda:0", dtype=torch.float32)
    dB = torch.randint(-8, 9, (K, N), generator=gen, device="cuda:0", dtype=torch.float32)
    dA[:, M] = float("inf")
    want = torch.cat([(dA[:, at:min(at + 200000, M)].double().t().contiguous() @ dB.double()).float() for at in range(0, M, 200000)])
    C = torch.empty((M, N), dtype=torch.float32, device="cuda:0")
    for key in b32.RING_KEYS[::2]:
        C.fill_(float("nan"))
        load(b32.library_for_key(key)).gemm(dA.data_ptr(), dB.data_ptr(), C.data_ptr(), M, N, K, M + 1, N, N)
        assert torch.equal(C, want), key


def test_results_stay_inside_their_rows():
    """lda, ldb and ldc beyond M and N, and a C off the vector alignment; neighbours keep what they held, and what lies in the padding
    of A and B (infinities) reaches no result."""
    rng = np.random.default_rng(6)
    A = np.full((72, 108), np.inf, np.float32)
    B = np.full((72, 96), np.inf, np.float32)
    A[:, :101] = rng.integers(-8, 9, (72, 101))
    B[:, :90] = rng.integers(-8, 9, (72, 90))
    exact = (A[:, :101].T.astype(np.int64) @ B[:, :90].astype(np.int64)).astype(np.float32)
    dA, dB = dev(A), dev(B)
    for key in b32.RING_KEYS:
        for ldc, offset in ((96, 0), (94, 2), (93, 1)):
            out = torch.full((101 * ldc + 16,), 7.0, dtype=torch.float32, device="cuda:0")
            load(b32.library_for_key(key)).gemm(dA.data_ptr(), dB.data_ptr(), out.data_ptr() + 4 * offset, 101, 90, 72, 108, 96, ldc)
            got = out.cpu().numpy()
            rows = got[offset:offset + 101 * ldc].reshape(101, ldc)
            assert np.array_equal(rows[:, :90], exact), (key, ldc)
            assert (rows[:, 90:] == 7).all() and (got[:offset] == 7).all() and (got[offset + 101 * ldc:] == 7).all(), (key, ldc)


def test_infinities_stay_in_their_row_and_column():
    """K off every step: what the copies do not fetch is zero, not what LDS held."""
    A = np.zeros((40, 71), np.float32)
    B = np.zeros((71, 50), np.float32)
    A[7, 70], B[70, 9] = np.inf, 1
    A[8, :], B[0, 9] = 1, 1
    want = np.zeros((40, 50), np.float32)
    want[7, :] = np.nan
    want[7, 9] = np.inf
    want[8, 9] = 2
    for key in b32.RING_KEYS:
        assert np.array_equal(run_sgemm_f32(load(b32.library_for_key(key)), A, B), want, equal_nan=True), key


def test_graph_replays_and_refusals():
    rng = np.random.default_rng(8)
    A, B = rng.integers(-8, 9, (200, 132)).astype(np.float32), rng.integers(-8, 9, (200, 92)).astype(np.float32)
    exact = A.T.astype(np.int64) @ B.astype(np.int64)
    dA, dB = dev(A), dev(B)
    lib = load(b32.library_for_key(b32.RING_KEYS[0]))
    C = torch.zeros((132, 92), dtype=torch.float32, device="cuda:0")
    args = (dA.data_ptr(), dB.data_ptr(), C.data_ptr(), 132, 92, 200, 132, 92, 92)
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
    assert lib.gemm(*args[:6], 130, *args[7:], check=False) == HELIX_ERR_INVALID_VALUE
    assert lib.gemm(dA.data_ptr() + 4, *args[1:], check=False) == HELIX_ERR_INVALID_VALUE
    conv = (dA.data_ptr(), dB.data_ptr(), C.data_ptr(), 1, 8, 8)
    assert lib.conv2d(*conv, 6, 8, 1, 1, 1, 0, check=False) == HELIX_ERR_UNSUPPORTED       # chunks across taps
    assert lib.conv2d(*conv, 4, 8, 4, 8, 1, 0, check=False) == HELIX_ERR_UNSUPPORTED       # 32 taps
    assert lib.conv2d(dA.data_ptr() + 4, *conv[1:], 8, 8, 1, 1, 1, 0, check=False) == HELIX_ERR_INVALID_VALUE


# batch, channels, H, W, filters, kH, kW, stride, pad
LAYERS = [(1, 4, 1, 1, 1, 1, 1, 1, 0),         # one pixel, one chunk
          (2, 32, 9, 11, 70, 3, 3, 1, 1),      # a tile is one tap; filters off 4
          (3, 12, 14, 10, 33, 5, 5, 2, 2),     # a tile over three taps
          (2, 64, 12, 12, 48, 5, 5, 1, 4),     # rows and columns of taps beyond the image
          (2, 100, 7, 7, 40, 1, 1, 1, 0),      # half a K tile left over
          (2, 4, 9, 12, 20, 5, 6, 1, 0),       # 30 taps, eight of them a tile
          (1, 8, 40, 3, 24, 31, 1, 3, 2),      # 31 taps
          (2, 96, 20, 23, 260, 3, 2, 3, 1)]    # several tiles both ways, rows off every multiple


@pytest.mark.parametrize("layer", LAYERS, ids=lambda l: "x".join(map(str, l)))
def test_every_configuration_convolves_integer_exact(layer):
    B, IC, H, W, OC, kH, kW, stride, pad = layer
    rng = np.random.default_rng(sum(layer))
    x = rng.integers(-4, 5, (B, H, W, IC)).astype(np.float32)
    w = rng.integers(-4, 5, (OC, kH, kW, IC)).astype(np.float32)
    want = O.conv2d_nhwc(x, w, stride, pad)
    for key in b32.RING_KEYS:
        assert np.array_equal(run_conv(load(b32.library_for_key(key)), x, w, stride, pad, torch.float32), want), key


def test_infinities_in_the_input_reach_their_pixels_only():
    """Padding, channels beyond the last tile and rows beyond the last pixel are zeros, not what lies beside them."""
    x = np.zeros((2, 6, 7, 20), np.float32)
    w = np.ones((35, 3, 3, 20), np.float32)
    x[0, 5, 6, 19] = np.inf
    want = np.zeros((2, 6, 7, 35), np.float32)
    want[0, 4:6, 5:7] = np.inf
    for key in b32.RING_KEYS:
        assert np.array_equal(run_conv(load(b32.library_for_key(key)), x, w, 1, 1, torch.float32), want), key


# batch, channels, H, W, filters, kH, kW, stride, pad: K = 75, 300, 800, 1200
EXACT_LAYERS = [(3, 3, 40, 40, 33, 5, 5, 2, 2), (2, 12, 20, 20, 33, 5, 5, 1, 2), (1, 32, 24, 24, 64, 5, 5, 1, 2), (1, 48, 20, 20, 96, 5, 5, 1, 2)]


@pytest.mark.parametrize("layer", EXACT_LAYERS, ids=lambda l: "x".join(map(str, l)))
def test_convolutions_are_as_exact_as_k_groups(layer):
    """The ring tiles and the family whose input stays in LDS, next to sgemm.hip's four and eight K groups."""
    B, IC, H, W, OC, kH, kW, stride, pad = layer
    rng = np.random.default_rng(sum(layer))
    x, w = rng.standard_normal((B, H, W, IC)).astype(np.float32), rng.standard_normal((OC, kH, kW, IC)).astype(np.float32)
    exact = np.zeros((B, *conv_out_hw(H, W, kH, kW, stride, pad), OC))
    xp = np.pad(x.astype(np.float64), ((0, 0), (pad, pad), (pad, pad), (0, 0)))
    for i in range(kH):
        for j in range(kW):
            exact += xp[:, i:, j:][:, :(exact.shape[1] - 1) * stride + 1:stride, :(exact.shape[2] - 1) * stride + 1:stride] @ w[:, i, j].T.astype(np.float64)
    keys = [k for k in b32.patch_keys() if c32.PATCH.layout((k[0], k[1], k[3], k[4], k[6]), *layer)] + (list(b32.RING_KEYS) if IC % 4 == 0 else [])

    def result(lib):
        dx, dw, dy = dev(x), dev(w), torch.empty(exact.shape, dtype=torch.float32, device="cuda:0")
        # without a workspace K is not partitioned beside; a channel count off 4 needs it for its copies
        wsb = lib.conv_workspace_bytes(B, H, W, IC, OC, kH, kW, stride, pad) if IC % 4 else 0
        ws = torch.empty(max(wsb, 16), dtype=torch.uint8, device="cuda:0")
        lib.conv2d(dx.data_ptr(), dw.data_ptr(), dy.data_ptr(), B, H, W, IC, OC, kH, kW, stride, pad, ws.data_ptr() if wsb else 0, wsb)
        return dy.cpu().numpy()

    errors = {}
    for c in b32.iter_kgroup_configs():
        errors[c[5]] = min(errors.get(c[5], 1.0), error(result(load(b32.sgemm_library(*c))), exact))
    for key in keys:
        # wave tiles of eight and more add a chain per K tile where channels are off 4, and are held to two groups there
        limit = errors[2] if IC % 4 and wave_tiles(key) >= 8 else min(errors[4], errors[8])
        assert error(result(load(b32.library_for_key(key))), exact) <= limit * scatter(exact.size), key
