"""Launches whose last round of tiles is partitioned along K (common/helix_tail.h): tile counts just above and far above a
multiple of 256, ragged edges in the partitioned tiles, K off the block; integer inputs, so every order of sums is exact."""
import numpy as np
import pytest
import torch

from utils.helix_runtime import load
from MI355X_FP32 import build_MI355X_FP32 as b32, MI355X_FP32_gemm as g32
from gpu_helpers import run_conv, run_sgemm_f32

pytestmark = pytest.mark.gpu


def ints(rng, shape, dtype):
    return rng.integers(-2, 3, shape).astype(dtype)


def exact_product(A, B):
    return A.astype(np.float64) @ B.astype(np.float64)      # whole numbers below 2^53


# (library, M, N, K): 257, 288, 260 and 258 tiles
F32 = [((64, 64, 32, 32, 32), 64 * 257, 64, 1152),
       ((64, 64, 32, 32, 32), 1500, 768, 2304),
       ((128, 64, 16, 32, 64), 2497, 830, 1031),
       ((128, 128, 16, 64, 32), 700, 5490, 777)]


@pytest.mark.parametrize("cfg,M,N,K", F32)
def test_sgemm_last_round_partitioned(cfg, M, N, K):
    lib = load(b32.sgemm_library(*cfg))
    key = b32.config_key(*cfg)
    tail, uniform = g32.tail_splits(key, M, N, K), g32.split_factor(key, M, N, K)
    tiles = -(-M // cfg[0]) * -(-N // cfg[1])
    assert tail >= 2
    assert lib.workspace_bytes(M, N, K) == max(tiles % 256 * tail * cfg[0] * cfg[1] * 4, uniform * M * N * 4 if uniform > 1 else 0)
    rng = np.random.default_rng(tiles)
    A, B = ints(rng, (M, K), np.float32), ints(rng, (K, N), np.float32)
    want = exact_product(A, B)
    assert np.array_equal(run_sgemm_f32(lib, A, B), want)
    assert np.array_equal(run_sgemm_f32(lib, A, B, workspace=False), want)


def test_conv_f32_last_round_partitioned():
    lib = load(b32.sgemm_library(64, 64, 32, 32, 32))
    batch, IC, H, W, OC = 9, 64, 43, 43, 63            # 261 tiles, ragged in both directions
    assert g32.tail_splits(b32.config_key(64, 64, 32, 32, 32), batch * H * W, OC, 9 * IC) >= 2
    rng = np.random.default_rng(3)
    x, w = ints(rng, (batch, H, W, IC), np.float32), ints(rng, (OC, 3, 3, IC), np.float32)
    got = run_conv(lib, x, w, 1, 1, torch.float32)
    want = torch.nn.functional.conv2d(torch.from_numpy(x).permute(0, 3, 1, 2), torch.from_numpy(w).permute(0, 3, 1, 2),
                                      padding=1).permute(0, 2, 3, 1).numpy()
    assert np.array_equal(got, want)
