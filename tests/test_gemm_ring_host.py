"""Ranking and selection of the four-wave tiles over a ring of LDS stages (MI355X_FP16/gemm_ring.hip, MI355X_FP32/gemm_ring.hip),
which have no profile, and the limits of their operands."""
import os
import subprocess

from utils import helix_runtime
from MI355X_FP16 import build_MI355X_FP16 as b16
from MI355X_FP16 import profile_MI355X_FP16 as p16
from MI355X_FP16 import MI355X_FP16_conv as c16
from MI355X_FP16 import MI355X_FP16_gemm as g16
from MI355X_FP32 import build_MI355X_FP32 as b32
from MI355X_FP32 import profile_MI355X_FP32 as p32
from MI355X_FP32 import MI355X_FP32_conv as c32
from MI355X_FP32 import MI355X_FP32_gemm as g32


def test_points_fit_the_template():
    assert len(set(b16.RING_KEYS)) == len(b16.RING_POINTS) == 25 and not set(b16.RING_KEYS) & set(p16.all_keys())
    for rows, cols, stages in b16.RING_POINTS:
        assert rows % 32 == cols % 32 == 0 and 32 <= rows <= 256 and 32 <= cols <= 256
        assert stages * (rows + cols) * 128 <= 160 * 1024 and (stages - 1) * (rows + cols) // 32 <= 63
        assert 4 * 16 * (cols + 16) <= stages * (rows + cols) * 128            # the strips that the results pass through
    key = b16.ring_key((224, 160, 3))
    assert key == (3, 224, 160, 112, 80, 0, 64, 3) and b16.is_ring_key(key) and not b16.is_dtl_key(key) and not b16.is_patch_key(key)
    assert b16.library_for_key(key).endswith("build/bin_fp16/libgemm_ring_3_224_160.so")
    assert b16.ring_job(key)[2] == {"K_STAGES": 3, "BLOCK_ROWS": 224, "BLOCK_COLS": 160}


def test_ranking_follows_the_rounds():
    """661 rows in three tiles of 224, and 207 tiles in one round of 256; few rows take small tiles."""
    assert b16.ring_key((224, 160, 3)) in g16.ring_ranked(661, 11008, 4096, 2)
    assert all(k[1] <= 64 for k in g16.ring_ranked(19, 1032, 952, 2))
    assert len(g16.ring_ranked(300, 8192, 4096)) == g16.RING_TOP
    seconds = lambda point: g16.ring_seconds(b16.ring_key(point), 8192, 8192, 8192, 3 * 8192 ** 2 * 2, g16.RING_GEMM)
    assert seconds((64, 64, 3)) > seconds((256, 128, 3))


def test_selection_times_the_family_and_keeps_its_winner(tmp_path, monkeypatch):
    """For products and for layers of whole chunks of channels; others are not offered to it."""
    monkeypatch.setattr(helix_runtime, "root_path", str(tmp_path))
    prof = {(2, 64, 64, 32, 32, 0, 64): 1e-5, (2, 128, 64, 64, 32, 0, 64): 2e-5}
    timed = []

    def run_config(k, M, N, K, **kw):
        timed.append(k)
        return 1e-6 if b16.is_ring_key(k) else 2e-6

    monkeypatch.setattr(g16, "run_config", run_config)
    key = g16.select_config(prof, 661, 1100, 4096)
    assert b16.is_ring_key(key) and set(prof) < set(timed) and len(set(timed)) == len(prof) + g16.RING_TOP
    timed.clear()
    assert g16.select_config(prof, 661, 1100, 4096) == key and not timed
    monkeypatch.setenv("HELIX_SELECTION", "model")
    assert g16.select_config(prof, 661, 1100, 4096) in prof
    monkeypatch.delenv("HELIX_SELECTION")

    class Library:
        def __init__(self, path):
            self.path = path

        def bench_conv(self, *a, **kw):
            return 0.0, 1e-6 if "gemm_ring" in self.path else 2e-6, 0.0

    monkeypatch.setattr(c16, "load", Library)
    assert b16.is_ring_key(c16.select_config(prof, 4, 64, 14, 14, 96, 1, 1, 1, 0))
    assert b16.is_ring_key(c16.select_config(prof, 4, 64, 14, 14, 96, 3, 3, 1, 1))
    assert not b16.is_ring_key(c16.select_config(prof, 4, 64, 14, 14, 96, 4, 8, 1, 1))
    assert not b16.is_ring_key(c16.select_config(prof, 4, 25, 14, 14, 96, 1, 1, 1, 0))


def test_fp32_family(tmp_path, monkeypatch):
    """The same of the FP32 family, which has two stages."""
    assert len(set(b32.RING_KEYS)) == len(b32.RING_POINTS) == 18 and not set(b32.RING_KEYS) & set(p32.all_keys())
    for rows, cols, waves_m in b32.RING_POINTS:
        assert waves_m in (1, 2, 4) and rows % (16 * waves_m) == cols % (64 // waves_m) == 0
        assert rows // waves_m <= 128 and cols * waves_m // 4 <= 128 and (rows + cols) * 256 + 1024 <= 160 * 1024
    key = b32.ring_key((64, 80, 4))
    assert key == (64, 80, 32, 16, 80, 2, 1, 0) and b32.is_ring_key(key) and not b32.is_patch_key(key)
    assert b32.library_for_key(key).endswith("build/bin_fp32/libgemm_ring_64_80_16_80.so")
    assert b32.ring_job(key)[2] == {"BLOCK_ROWS": 64, "BLOCK_COLS": 80, "WAVES_M": 4}
    assert b32.ring_key((64, 64, 2)) in g32.ring_ranked(4000, 2300, 770)
    assert b32.ring_key((64, 80, 4)) in g32.ring_ranked(283256, 72, 331, 1)
    monkeypatch.setattr(helix_runtime, "root_path", str(tmp_path))
    prof = {b32.config_key(64, 64, 16, 32, 32): 1.0, b32.config_key(128, 64, 16, 32, 32): 1.7}
    timed = []
    monkeypatch.setattr(g32, "run_config", lambda k, M, N, K, **kw: timed.append(k) or (1e-6 if b32.is_ring_key(k) else 2e-6))
    key = g32.select_config(prof, 661, 1100, 4096)
    assert b32.is_ring_key(key) and set(prof) < set(timed) and len(set(timed)) == len(prof) + g32.RING_TOP
    timed.clear()
    assert g32.select_config(prof, 661, 1100, 4096) == key and not timed
    assert g32.verified_config(prof, 661, 1100, 4096, families=False) in prof

    class Library:
        def __init__(self, path):
            self.path = path

        def bench_conv(self, *a, **kw):
            return 0.0, 1e-6 if "gemm_ring" in self.path else 2e-6, 0.0

    monkeypatch.setattr(c32, "load", Library)
    assert b32.is_ring_key(c32.select_config(prof, 4, 64, 28, 28, 96, 3, 3, 1, 1))
    assert not c32.ring_ranked((4, 25, 28, 28, 96, 3, 3, 1, 1)) and not c32.ring_ranked((4, 64, 28, 28, 96, 11, 11, 1, 5))
    assert len(c32.ring_ranked((4, 4, 28, 28, 96, 5, 6, 1, 0))) == g32.RING_CONV_TOP


def test_few_rows_of_long_k_are_left_to_the_others(monkeypatch):
    """Decode products: a selection neither ranks nor times the ring tiles, which are never ahead there."""
    for g, build, prof, problem in ((g16, b16, {(2, 64, 64, 32, 32, 0, 64): 1e-5}, (16, 28672, 8192)),
                                    (g32, b32, {b32.config_key(64, 64, 16, 32, 32): 1.0}, (4, 11008, 4096))):
        timed = []
        monkeypatch.setattr(g, "run_config", lambda k, *a, **kw: timed.append(k) or 1e-6)
        assert g.verified_config(prof, *problem) in prof
        assert set(timed) == set(prof) and not any(build.is_ring_key(k) for k in timed)
        assert len(g.ring_ranked(17, 4096, 4096)) == len(g.ring_ranked(16, 4096, 1016)) == len(g.ring_ranked(30000, 16, 2000)) == g.RING_TOP


def test_zeros_are_read_beyond_every_operand(tmp_path):
    """The offset of what a copy has not got lies behind a K tile of the largest operand that the FP32 tiles take, 4 GiB, aligned as a
    copy is."""
    exe, key = str(tmp_path / "check"), b32.ring_key((32, 64, 2))
    defines = [f"-D{k}={v}" for k, v in b32.ring_job(key)[2].items()]
    build = subprocess.run(["hipcc", "-O1", "-w", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                            f"-I{helix_runtime._find_include_dir()}", f"-I{os.path.join(helix_runtime.SRC_ROOT, 'common')}",
                            f"-I{os.path.join(helix_runtime.SRC_ROOT, 'MI355X_FP32')}", *defines,
                            os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "gemm_ring_check.cpp"), "-o", exe],
                           capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-2000:]
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout[-200:]
