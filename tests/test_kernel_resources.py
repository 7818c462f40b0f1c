"""Register spills of the built kernels, as the compiler reported them (resource_usage.json beside the libraries)."""
import pytest

from utils.helix_runtime import kernel_resources
from MI355X_FP16 import build_MI355X_FP16 as b16
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


def test_fp16_kernels_that_spill():
    """The tile kernels (modes: 0 GEMM, 1 general gather, 2 gather inside one filter tap) that the compiler finds no
    registers for, and how many bytes per lane they spill at most; the selection passes over such a gather, and every
    configuration that is not listed here stays available in all three modes."""
    known = {(2, 128, 128, 128, 128, 64): (0, 240, 32), (2, 128, 48, 128, 48, 128): (0, 112, 0),
             (2, 128, 64, 128, 64, 128): (0, 784, 52), (2, 128, 96, 128, 96, 128): (304, 1104, 892),
             (2, 256, 256, 128, 64, 64): (0, 32, 0), (2, 256, 256, 64, 128, 64): (0, 32, 0),
             (3, 128, 192, 64, 48, 128): (0, 0, 228), (3, 256, 128, 64, 64, 64): (0, 0, 36),
             (3, 256, 64, 64, 32, 128): (0, 0, 52), (3, 64, 256, 32, 64, 128): (0, 0, 52)}
    for split_k, family in ((0, "gemm"), (1, "gemm_splitK")):
        for cfg in b16.iter_configs(split_k):
            for mode, most in enumerate(known.get(cfg, (0, 0, 0)) if not split_k else (0, 0, 0)):
                found = scratch(b16.kernel_library(family, *cfg), f"helix_gemm_f16_kernelILi{mode}E")
                assert len(found) == 1 and found[0] <= most, (family, cfg, mode, found)
