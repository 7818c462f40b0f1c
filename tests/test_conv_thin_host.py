"""Host side of the thin-input convolution (common/helix_conv_thin.h), compiled and run on the CPU."""
import os
import random
import subprocess

import pytest

from utils.helix_runtime import SRC_ROOT, _find_include_dir
from utils.hip_ctypes import HELIX_ERR_INVALID_VALUE, HelixError
from MI355X_FP16 import MI355X_FP16_conv as c16

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


def layers():
    rng = random.Random(5)
    out = [(32, 3, 224, 224, 64, 7, 7, 2, 3), (1, 1, 40, 300, 32, 11, 20, 2, 0), (1, 3, 7, 20000, 64, 7, 7, 1, 3),
           (600, 3, 7, 20000, 64, 7, 7, 1, 3), (1, 4, 1, 2 ** 28 - 2, 8, 1, 1, 1, 0), (1, 4, 1, 2 ** 28 - 1, 8, 1, 1, 1, 0),
           (1, 3, 224, 224, 768, 16, 16, 16, 0), (1, 5, 9, 9, 8, 3, 3, 1, 1), (1, 8, 9, 9, 8, 3, 3, 1, 1),
           (1, 1, 3, 3, 64 * 65535, 3, 3, 1, 1), (1, 1, 3, 3, 64 * 65535 + 1, 3, 3, 1, 1)]
    while len(out) < 3000:
        kH, kW = rng.randint(1, 14), rng.randint(1, 30)
        H, W = rng.randint(kH, 60), rng.choice((rng.randint(kW, 100), rng.randint(kW, 12000)))
        out.append((rng.choice((1, 2, 9, 40, 600)), rng.randint(1, 4), H, W, rng.choice((8, 64, 70, 1000)), kH, kW,
                    rng.randint(1, 5), rng.randint(0, max(kH, kW))))
    return out


def test_host_knows_which_layers_the_thin_kernel_takes(check):
    cases = layers()
    run = subprocess.run([check, "plans"], input="\n".join(" ".join(map(str, l)) for l in cases), capture_output=True, text=True)
    taken = [line == "1" for line in run.stdout.split()]
    assert len(taken) == len(cases) and 500 < sum(taken) < 2900
    assert [c16.runs_thin(*l) for l in cases] == taken


@pytest.mark.parametrize("layer", [(1, 3, 5, 5, 8, 7, 7, 3, 0), (1, 3, 9, 5, 8, 7, 7, 2, 0), (1, 1, 3, 30, 8, 5, 5, 1, 0)])
def test_filter_beyond_the_image_is_still_refused_by_the_selection(layer, monkeypatch):
    class Library:
        def bench_conv(self, *a, **kw):
            raise HelixError("helix_bench_conv", HELIX_ERR_INVALID_VALUE)
    assert not c16.runs_thin(*layer)
    monkeypatch.setattr(c16, "load", lambda path: Library())
    with pytest.raises(RuntimeError, match="none of"):
        c16.verified_config({(2, 64, 64, 32, 32, 0, 64): 1e-5}, *layer)


def test_selection_of_a_thin_layer_times_nothing(monkeypatch):
    """The libraries' thin kernels are one and the same: the pick is the model's first one without K partitions, whose
    workspace holds no partial sums."""
    prof = {k: 1e-5 * (i + 1) for i, k in enumerate([(2, 32, 64, 32, 32, 1, 64), (2, 64, 64, 32, 32, 1, 64),
                                                     (2, 128, 64, 64, 32, 0, 64), (2, 64, 64, 32, 32, 0, 64)])}
    monkeypatch.setattr(c16, "load", lambda path: pytest.fail("a library was loaded to be timed"))
    layer = (1, 3, 30, 30, 64, 7, 7, 2, 3)
    ranked = c16.ranked_configs(prof, 15 * 15, 64, 8 * 49, 8)
    assert ranked[0][5] == 1
    assert c16.verified_config(prof, *layer) == next(k for k in ranked if k[5] == 0)
    with pytest.raises(BaseException, match="a library was loaded"):
        c16.verified_config(prof, 1, 8, 30, 30, 64, 7, 7, 2, 3)
