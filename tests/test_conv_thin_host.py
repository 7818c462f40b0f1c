"""Host side of the thin-input convolution (common/helix_conv_thin.h), compiled and run on the CPU."""
import os
import subprocess

import pytest

from utils.helix_runtime import SRC_ROOT, _find_include_dir

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("conv_thin") / "conv_thin_check")
    build = subprocess.run(["hipcc", "-O1", "-w", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                            "-packed-fp32-ops", f"-I{_find_include_dir()}", f"-I{os.path.join(SRC_ROOT, 'common')}",
                            os.path.join(HERE, "cpp", "conv_thin_check.cpp"), "-o", exe], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-2000:]
    return exe


def test_staging_loads_stay_inside_the_input(check):
    """Also where x has an odd number of halves: no load reaches into the dword that holds the last of them."""
    run = subprocess.run([check, "windows"], capture_output=True, text=True)
    assert run.returncode == 0 and "mismatches 0" in run.stdout, run.stdout + run.stderr
