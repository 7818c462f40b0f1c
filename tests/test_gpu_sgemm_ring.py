"""FP32 products on four-wave tiles over a ring of LDS stages (MI355X_FP32/gemm_ring.hip): every configuration at the edges of its
tiles, through the C ABI."""
import numpy as np
import pytest
import torch

from utils.helix_runtime import load
from utils.hip_ctypes import HELIX_ERR_INVALID_VALUE, HELIX_ERR_UNSUPPORTED
from MI355X_FP32 import build_MI355X_FP32 as b32
from gpu_helpers import dev, run_sgemm_f32

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


def test_the_bits_of_sgemm():
    """Products of a result are added in ascending k, each rounded, as in an unpartitioned launch of sgemm.hip."""
    rng = np.random.default_rng(4)
    A, B = rng.standard_normal((290, 777)).astype(np.float32), rng.standard_normal((777, 301)).astype(np.float32)
    want = run_sgemm_f32(load(b32.default_library()), A, B, workspace=False)
    for key in b32.RING_KEYS:
        assert np.array_equal(run_sgemm_f32(load(b32.library_for_key(key)), A, B), want), key


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
    assert lib.conv2d(dA.data_ptr(), dB.data_ptr(), C.data_ptr(), 1, 4, 4, 8, 8, 1, 1, 1, 0, check=False) == HELIX_ERR_UNSUPPORTED
