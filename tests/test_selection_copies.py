"""The copies of the weights that a selection is timed on (MI355X_FP16_gemm.verified_config)."""
import pytest

from utils.hip_ctypes import HelixError
from MI355X_FP16 import MI355X_FP16_gemm as g16

A, B = (2, 256, 256, 128, 64, 0, 64), (2, 128, 128, 64, 64, 0, 64)
PROFILE = {A: 1e-4, B: 5e-5}
CACHE = 256 << 20


@pytest.mark.parametrize("N,K", [(4096, 4096), (8192, 4096 - 8), (8192, 4096), (11008, 4096), (8192, 8192), (16384, 8192 - 8),
                                 (16384, 8192), (28672, 8192), (60000, 40001)])
def test_copies_fill_the_cache_and_no_more(N, K, monkeypatch):
    seen = set()
    monkeypatch.setattr(g16, "run_config", lambda k, M, N, K, warmup, iters, copies=1: seen.add(copies) or 1e-4)
    g16.verified_config(PROFILE, 661, N, K)
    (copies,) = seen
    weights = N * g16.padded_k(K) * 2
    if weights < 64 << 20:
        assert copies == 1
    else:
        assert copies * weights >= CACHE and (copies - 1) * weights < CACHE     # what they add is bounded


def test_problem_whose_copies_do_not_fit_is_selected_on_one(monkeypatch):
    def run_config(k, M, N, K, warmup, iters, copies=1):
        if copies > 1:
            raise HelixError("helix_bench", 2)                                  # out of memory
        return {A: 2e-4, B: 1e-4}[k]
    monkeypatch.setattr(g16, "run_config", run_config)
    assert g16.verified_config(PROFILE, 661, 11008, 4096) == B


def test_problem_nothing_can_run_is_refused(monkeypatch):
    def run_config(*a, **kw):
        raise HelixError("helix_bench", 1)
    monkeypatch.setattr(g16, "run_config", run_config)
    with pytest.raises(RuntimeError, match="661x11008x4096"):
        g16.verified_config(PROFILE, 661, 11008, 4096)
