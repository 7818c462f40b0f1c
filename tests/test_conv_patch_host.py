"""Host side of the convolutions whose input stays in LDS (common/helix_conv_patch.h), compiled and run on the CPU."""
import os
import random
import subprocess

import pytest

from utils.helix_runtime import SRC_ROOT, _find_include_dir
from utils import helix_runtime
from utils.hip_ctypes import HELIX_ERR_UNSUPPORTED, HelixError
from MI355X_FP16 import build_MI355X_FP16 as b16
from MI355X_FP16 import MI355X_FP16_conv as c16
from MI355X_FP32 import build_MI355X_FP32 as b32
from MI355X_FP32 import MI355X_FP32_conv as c32

HERE = os.path.dirname(os.path.abspath(__file__))


def layers():
    rng = random.Random(3)
    out = [(4, 256, 14, 14, 256, 3, 3, 1, 1), (1, 8, 1, 1, 1, 1, 1, 1, 0), (1, 8, 5, 5, 8, 3, 3, 1, 9), (1, 12, 9, 9, 8, 3, 3, 1, 1),
           (3, 8, 9, 9, 8, 2, 2, 5, 0), (1, 2048, 40, 40, 64, 3, 3, 1, 1), (2, 8, 7, 7, 8, 9, 9, 1, 0), (900, 8, 96, 97, 4, 3, 3, 1, 1)]
    while len(out) < 1500:
        out.append((rng.randint(1, 9), rng.choice((8 * rng.randint(1, 30), 8 * rng.randint(1, 30), rng.randint(1, 60))), rng.randint(1, 40), rng.randint(1, 40), rng.randint(1, 300),
                    rng.randint(1, 7), rng.randint(1, 7), rng.randint(1, 5), rng.randint(0, 5)))
    return out


@pytest.mark.parametrize("build,conv,precision,index", [(b16, c16, "FP16", 0), (b16, c16, "FP16", 10), (b16, c16, "FP16", 21),
                                                        (b32, c32, "FP32", 1), (b32, c32, "FP32", 13), (b32, c32, "FP32", 20)])
def test_plans_stay_in_bounds_and_match_the_host_model(build, conv, precision, index, tmp_path):
    """Every block of every layer writes and reads inside the LDS that its plan reserves; the host model, which ranks the
    configurations, has the same bytes and workgroups and refuses the same layers."""
    exe = str(tmp_path / "check")
    point = build.PATCH_POINTS[index]
    defines = [f"-D{k}={v}" for k, v in build.patch_job(build.patch_key(point))[2].items()]
    build = subprocess.run(["hipcc", "-O1", "-w", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                            f"-I{_find_include_dir()}", f"-I{os.path.join(SRC_ROOT, 'common')}", f"-I{os.path.join(SRC_ROOT, 'MI355X_' + precision)}",
                            *defines, os.path.join(HERE, "cpp", "conv_patch_check.cpp"), "-o", exe], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-2000:]
    cases = layers()
    run = subprocess.run([exe], input="\n".join(" ".join(map(str, l)) for l in cases), capture_output=True, text=True)
    assert run.returncode == 0, run.stdout[-200:]
    got = [None if line == "none" else tuple(map(int, line.split())) for line in run.stdout.splitlines()]
    assert len(got) == len(cases) and 200 < sum(g is not None for g in got) < len(cases)
    assert [conv.PATCH.layout(point, *l) for l in cases] == got


def test_family_is_ranked_for_the_layers_it_can_run():
    layer = (4, 256, 14, 14, 256, 3, 3, 1, 1)
    ranked = c16.patch_ranked(layer)
    assert len(ranked) == c16.PATCH_TOP and all(b16.is_patch_key(k) and not b16.is_dtl_key(k) for k in ranked)
    assert ranked == [b16.patch_key(p) for p in sorted(b16.PATCH_POINTS, key=lambda p: (c16.PATCH.seconds(p, *layer), p))[:c16.PATCH_TOP]]
    assert c16.patch_ranked((4, 12, 14, 14, 256, 3, 3, 1, 1)) == []         # channels off the 16-byte chunk
    assert c16.patch_ranked((4, 4096, 64, 64, 256, 3, 3, 1, 1)) == []       # rows beyond LDS
    assert c16.patch_ranked((1, 8, 3, 30, 8, 5, 5, 1, 0)) == [] == c32.patch_ranked((1, 8, 3, 30, 8, 5, 5, 1, 0))   # a filter beyond the image
    assert all(b32.is_patch_key(k) for k in c32.patch_ranked((4, 3, 14, 14, 256, 3, 3, 1, 1))) and len(b32.patch_keys()) == 22
    assert not any(b32.is_patch_key(b32.config_key(*c)) for c in list(b32.iter_configs()) + list(b32.iter_kgroup_configs()))
    assert not b32.is_patch_key((4, 128, 0, 0, 0, 0, 4, 4))                 # the GEMV rows
    assert b32.library_for_key((80, 32, 32, 80, 16, 0, 4, 4)).endswith("build/bin_fp32/libconv_patch_80_32_80_16_4.so")
    assert b16.library_for_key((2, 32, 16, 32, 16, 8, 64, 2)).endswith("build/bin_fp16/libconv_patch_32_16_32_16_8.so")


def test_selection_times_the_family_and_keeps_its_winner(tmp_path, monkeypatch):
    """The first few configurations of the family are timed beside the profiled ones; a winner among them is recorded and
    handed out again though no profile holds it."""
    monkeypatch.setattr(helix_runtime, "root_path", str(tmp_path))
    prof = {(2, 64, 64, 32, 32, 0, 64): 1e-5, (2, 128, 64, 64, 32, 0, 64): 2e-5}
    timed = []

    class Library:
        def __init__(self, path):
            self.path = path

        def bench_conv(self, *a, **kw):
            timed.append(os.path.basename(self.path))
            if "_8." in self.path:
                raise HelixError("helix_bench_conv", HELIX_ERR_UNSUPPORTED)
            return 0.0, 1e-6 if "conv_patch" in self.path else 2e-6, 0.0

    monkeypatch.setattr(c16, "load", Library)
    layer = (4, 64, 14, 14, 64, 3, 3, 1, 1)
    key = c16.select_config(prof, *layer)
    assert b16.is_patch_key(key) and key in c16.patch_ranked(layer) and key[5] != 8
    assert {"libgemm_2_64_64_32_32_64.so", "libgemm_2_128_64_64_32_64.so"} < set(timed)
    timed.clear()
    assert c16.select_config(prof, *layer) == key and not timed
    monkeypatch.setenv("HELIX_SELECTION", "model")
    assert c16.select_config(prof, *layer) in prof
