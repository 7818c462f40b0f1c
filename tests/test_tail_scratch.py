"""The partial tiles of a partitioned last round (common/helix_tail.h) against the static scratch array: the entry point
that has nothing but that array sums in the same order as a launch with the workspace, whatever the shape."""
import math
import random

import pytest
import torch

from utils import seeded_inputs
from utils.helix_runtime import load
from utils.hip_ctypes import STATIC_SCRATCH_BYTES
from MI355X_FP32 import build_MI355X_FP32 as b32, MI355X_FP32_gemm as g32

# (configuration, M, N, K): the choice without a limit takes 87 tiles * 5 pieces * 64 KB = 27 MB in the first
SHAPES = [((128, 128, 32, 64, 32), 5638, 2414, 1621), ((64, 64, 32, 32, 32), 1500, 768, 2304)]


def tail_bytes(key, M, N, K):
    tiles = math.ceil(M / key[0]) * math.ceil(N / key[1])
    return tiles % 256 * g32.tail_splits(key, M, N, K) * key[0] * key[1] * 4


def test_last_round_partials_fit_the_static_scratch():
    rng = random.Random(3)
    shapes = [(cfg, M, N, K) for cfg, M, N, K in SHAPES]
    configs = list(b32.iter_configs())
    for _ in range(3000):
        shapes.append((rng.choice(configs), int(math.exp(rng.uniform(4, 10))), int(math.exp(rng.uniform(4, 9.4))),
                       rng.randint(256, 4096)))
    partitioned = 0
    for cfg, M, N, K in shapes:
        need = tail_bytes(b32.config_key(*cfg), M, N, K)
        partitioned += need > 0
        assert need <= STATIC_SCRATCH_BYTES, (cfg, M, N, K)
    assert partitioned > 20


@pytest.mark.gpu
@pytest.mark.parametrize("cfg,M,N,K", SHAPES)
def test_static_scratch_gives_the_workspace_bits(cfg, M, N, K):
    lib = load(b32.sgemm_library(*cfg))
    ld_a, ld_b = -(-M // 4) * 4, -(-N // 4) * 4
    A = torch.zeros((K, ld_a), device="cuda:0")
    B = torch.zeros((K, ld_b), device="cuda:0")
    A[:, :M] = torch.from_numpy(seeded_inputs.uniform_pm1((K, M), seeded_inputs.SEED_A))
    B[:, :N] = torch.from_numpy(seeded_inputs.uniform_pm1((K, N), seeded_inputs.SEED_B))
    want, got = torch.full((2, M, N), float("nan"), device="cuda:0")
    wsb = lib.workspace_bytes(M, N, K)
    assert wsb == max(tail_bytes(b32.config_key(*cfg), M, N, K), uniform_bytes(cfg, M, N, K)) > 0
    ws = torch.empty(wsb, dtype=torch.uint8, device="cuda:0")
    stream = torch.cuda.current_stream().cuda_stream
    lib.gemm(A.data_ptr(), B.data_ptr(), want.data_ptr(), M, N, K, ld_a, ld_b, N, ws.data_ptr(), wsb, stream)
    lib.gemm_static_scratch(A.data_ptr(), B.data_ptr(), got.data_ptr(), M, N, K, ld_a, ld_b, N, stream)
    torch.cuda.synchronize()
    assert not torch.isnan(want).any() and torch.equal(want, got)


def uniform_bytes(cfg, M, N, K):
    s = g32.split_factor(b32.config_key(*cfg), M, N, K)
    return s * M * N * 4 if s > 1 else 0
