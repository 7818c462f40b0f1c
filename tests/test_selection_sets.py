"""The sets of operands that a selection's launches take in turn (utils.helix_runtime.operand_sets)."""
import pytest

from utils import helix_runtime, hip_ctypes
from MI355X_FP16 import build_MI355X_FP16 as b16
from MI355X_FP16 import MI355X_FP16_conv as c16
from MI355X_FP16 import MI355X_FP16_gemm as g16
from MI355X_FP32 import build_MI355X_FP32 as b32
from MI355X_FP32 import MI355X_FP32_conv as c32
from MI355X_FP32 import MI355X_FP32_gemm as g32

PROF16 = {(2, 64, 64, 32, 32, 0, 64): 1e-5, (2, 128, 64, 64, 32, 0, 64): 2e-5}
PROF32 = {b32.config_key(64, 64, 16, 32, 32): 1.0, b32.config_key(128, 64, 16, 32, 32): 1.7}
# m, n, k: sets in turn, also where the memory-side cache is full of one; beyond a GiB; FP16 weights that are copied instead
PRODUCTS = [((269, 2376, 1376), 3, 3), ((127619, 5, 458), 3, 3), ((8192, 8192, 8192), 1, 3), ((40, 28672, 8192), 3, 3),
            ((32768, 32768, 8192), 1, 1), ((661, 11008, 4096), 1, 3)]
LAYERS = [((32, 64, 56, 56, 64, 3, 3, 1, 1), 3), ((64, 64, 150, 150, 64, 1, 1, 1, 0), 3), ((256, 64, 150, 150, 64, 1, 1, 1, 0), 1)]


def libraries(monkeypatch, modules, ring_seconds, room=True):
    """Libraries whose ring tiles take `ring_seconds` and all others 1 s; what they are asked to time.  Without `room` the device holds
    one set of operands and no more."""
    asked = []

    def answer(sets, rotate_bytes, seconds):
        asked.append((sets, rotate_bytes))
        if not room and (sets > 1 or rotate_bytes):
            raise hip_ctypes.HelixError("helix_bench_sets", 2)          # out of memory
        return seconds, seconds, seconds

    class Library:
        def __init__(self, path):
            self.seconds = ring_seconds if "gemm_ring" in path else 1.0

        def bench(self, M, N, K, warmup, iters, outer=1, rotate_bytes=0, sets=1):
            return answer(sets, rotate_bytes, self.seconds)

        def bench_conv(self, *layer, warmup, iters, sets=1):
            return answer(sets, 0, self.seconds)

    for module in modules:
        monkeypatch.setattr(module, "load", Library)
    return asked


@pytest.mark.parametrize("problem,sets16,sets32", PRODUCTS)
def test_products_are_timed_on_sets_in_turn(problem, sets16, sets32, monkeypatch):
    asked = libraries(monkeypatch, (g16, g32), 0.99)
    assert b16.is_ring_key(g16.verified_config(PROF16, *problem))         # a hundredth ahead is ahead
    copies = g16.weight_copies(*problem[1:])
    assert {s for s, _ in asked} == {sets16} and {bool(r) for _, r in asked} == {copies > 1}
    asked.clear()
    assert b32.is_ring_key(g32.verified_config(PROF32, *problem))
    assert set(asked) == {(sets32, 0)}


@pytest.mark.parametrize("layer,sets", LAYERS)
def test_layers_are_timed_on_sets_in_turn(layer, sets, monkeypatch):
    asked = libraries(monkeypatch, (c16, c32), 0.99)
    assert b16.is_ring_key(c16.verified_config(PROF16, *layer)) and b32.is_ring_key(c32.verified_config(PROF32, *layer))
    assert set(asked) == {(sets, 0)}


@pytest.mark.parametrize("problem", [p[0] for p in PRODUCTS])
def test_products_whose_sets_do_not_fit_are_timed_on_one(problem, monkeypatch):
    asked = libraries(monkeypatch, (g16, g32), 0.99, room=False)
    for verified_config, prof, is_ring in ((g16.verified_config, PROF16, b16.is_ring_key), (g32.verified_config, PROF32, b32.is_ring_key)):
        assert is_ring(verified_config(prof, *problem)) and asked[-1] == (1, 0)


@pytest.mark.parametrize("layer", [l[0] for l in LAYERS])
def test_layers_whose_sets_do_not_fit_are_timed_on_one(layer, monkeypatch):
    asked = libraries(monkeypatch, (c16, c32), 0.99, room=False)
    assert b16.is_ring_key(c16.verified_config(PROF16, *layer)) and b32.is_ring_key(c32.verified_config(PROF32, *layer))
    assert asked[-1] == (1, 0)


def test_rows_of_the_reports_are_timed_on_one_set(monkeypatch):
    asked = libraries(monkeypatch, (g16, g32), 0.99)
    g16.run_config((2, 64, 64, 32, 32, 0, 64), 269, 2376, 1376)
    g32.run_config(b32.config_key(64, 64, 16, 32, 32), 269, 2376, 1376)
    assert asked == [(1, 0), (1, 0)]


def test_candidates_of_a_selection_share_their_buffers():
    """All passes of one selection, and nothing outside it; the next selection has buffers of its own, also after an error."""
    seen = []

    def time_config(k, warmup, iters):
        seen.append(hip_ctypes._buffers.get())
        if k == "c":
            raise RuntimeError("cannot run")
        return {"a": 1.0, "b": 1.01}[k]

    assert helix_runtime.fastest_of(["a", "b", "c"], time_config, "p") == "a" and hip_ctypes._buffers.get() is None
    assert len(seen) == 7 and seen[0] is not None and len({id(s) for s in seen}) == 1
    with pytest.raises(RuntimeError):
        helix_runtime.fastest_of(["c"], time_config, "p")
    assert hip_ctypes._buffers.get() is None and seen[-1] is not seen[0] and seen[-1] is not None


def test_leaders_are_timed_until_the_device_has_come_to_rest():
    """Two rounds, and more while the fastest of a round is ahead of all before it; six at most."""
    def picks(times):
        left = {k: list(t) for k, t in times.items()}
        pick = helix_runtime.fastest_of(list(times), lambda k, warmup, iters: 1.0 if iters == 5 else left[k].pop(0), "p")
        return pick, {len(times[k]) - len(left[k]) for k in times}

    assert picks({"a": [1.2, 1.1, 1.0, 1.0, 0.1], "b": [1.3, 1.12, 0.97, 0.965, 2.0]}) == ("b", {4})
    assert picks({"a": [1.0, 0.995, 0.1], "b": [1.01, 1.0, 0.1]}) == ("a", {2})
    assert picks({"a": [2.0 ** -i for i in range(9)], "b": [1.1 * 2.0 ** -i for i in range(9)]}) == ("a", {6})


def test_sets_end_at_a_gib():
    assert helix_runtime.operand_sets(1) == helix_runtime.OPERAND_SETS == 3
    assert helix_runtime.operand_sets((1 << 30) - 1) == 3 and helix_runtime.operand_sets(1 << 30) == 1
