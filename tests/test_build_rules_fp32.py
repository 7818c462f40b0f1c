"""build_MI355X_FP32.is_valid_config against the FP32 template's own static_asserts."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from utils.helix_runtime import SRC_ROOT, _find_include_dir
from MI355X_FP32 import build_MI355X_FP32 as b32


def compiles(BM, BN, BK, WAVE_M, WAVE_N, KG):
    defines = dict(BM=BM, BN=BN, BK=BK, WAVE_M=WAVE_M, WAVE_N=WAVE_N, K_GROUPS=KG)
    cmd = ["hipcc", "-std=c++17", "--offload-arch=gfx950", "--cuda-host-only", "-fsyntax-only", "-w", f"-I{_find_include_dir()}",
           f"-I{os.path.join(SRC_ROOT, 'common')}"] + [f"-D{k}={v}" for k, v in defines.items()]
    return subprocess.run(cmd + [f"{SRC_ROOT}/MI355X_FP32/sgemm.hip"], capture_output=True).returncode == 0


# (BMt, BNt, BK, WAVE_M, WAVE_N, K_GROUPS): K tiles of no power of two, of one chunk, shares of less than two chunks per wave
# group, rows of more chunks than the fragments' rows can swizzle over, LDS beyond a compute unit's
@pytest.mark.parametrize("point", [(1, 1, 24, 32, 32, 1), (1, 1, 4, 32, 32, 1), (1, 1, 32, 32, 32, 8), (1, 1, 256, 32, 32, 8),
                                   (2, 2, 128, 64, 64, 1)], ids=lambda p: "_".join(map(str, p)))
def test_points_the_template_refuses_are_not_built(point):
    BMt, BNt, BK, WAVE_M, WAVE_N, KG = point
    assert not compiles(BMt * WAVE_M, BNt * WAVE_N, BK, WAVE_M, WAVE_N, KG)
    assert not b32.is_valid_config(BMt, BNt, BMt * WAVE_M, BNt * WAVE_N, BK, WAVE_M, WAVE_N, KG)


def test_points_at_the_edges_of_the_rules_compile():
    points = [(1, 1, 8, 32, 32, 1), (1, 1, 128, 32, 32, 8), (1, 1, 128, 32, 32, 16), (2, 2, 64, 32, 32, 4), (4, 2, 32, 64, 128, 1)]
    for BMt, BNt, BK, WAVE_M, WAVE_N, KG in points:
        assert b32.is_valid_config(BMt, BNt, BMt * WAVE_M, BNt * WAVE_N, BK, WAVE_M, WAVE_N, KG)
    with ThreadPoolExecutor(4) as ex:
        built = list(ex.map(lambda p: compiles(p[0] * p[3], p[1] * p[4], *p[2:]), points))
    assert all(built)
