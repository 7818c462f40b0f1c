"""Register spills of the built kernels, as the compiler reported them (resource_usage.json beside the libraries)."""
import pytest

from utils.helix_runtime import kernel_resources
from MI355X_FP32 import build_MI355X_FP32 as b32


def scratch(library, kernel):
    """Scratch bytes per lane of the kernels of a library whose name contains `kernel`."""
    usage = kernel_resources(library)
    if not usage:
        pytest.skip("libraries not built here")
    return [res["scratch"] for name, res in usage.items() if kernel in name]


def test_fp32_kernels_do_not_spill():
    """Nor the convolution kernels, which the selection ranks by their GEMM times; 128 x 128 wave tiles with BK = 32 (256
    accumulators and 64 or more staging registers per lane) are the exception in both modes."""
    configs = [c + (1,) for c in b32.iter_configs()] + list(b32.iter_kgroup_configs())
    for BM, BN, BK, WAVE_M, WAVE_N, KG in configs:
        if (WAVE_M, WAVE_N, BK) == (128, 128, 32):
            continue
        found = scratch(b32.sgemm_library(BM, BN, BK, WAVE_M, WAVE_N, KG), "helix_sgemm_f32_kernel")
        assert found == [0, 0], (BM, BN, BK, WAVE_M, WAVE_N, KG)
