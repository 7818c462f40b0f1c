"""FP16 convolutions through the workspace, and what is refused of it."""
import numpy as np
import pytest
import torch

from utils.helix_runtime import load
from utils.hip_ctypes import HELIX_ERR_INVALID_VALUE
from MI355X_FP16 import build_MI355X_FP16 as b16
from oracle import oracle as O
from gpu_helpers import dev

pytestmark = pytest.mark.gpu

LIBS = [("gemm", 2, 64, 64, 32, 32, 64), ("gemm_splitK", 2, 64, 64, 32, 32, 64), ("gemm", 2, 128, 64, 64, 32, 128)]


def integers(layer):
    """Inputs in {-1, 0, 1} and the result, a whole number below 2048: exact in any order of the sums."""
    batch, IC, H, W, OC, kH, kW, stride, pad = layer
    rng = np.random.default_rng(sum(layer))
    x = rng.integers(-1, 2, (batch, H, W, IC)).astype(np.float16)
    w = rng.integers(-1, 2, (OC, kH, kW, IC)).astype(np.float16)
    want = O.conv2d_nhwc(x.astype(np.float32), w.astype(np.float32), stride, pad)
    assert np.abs(want).max() < 2048
    return x, w, want


@pytest.mark.parametrize("IC", [1, 3, 6])
def test_workspace_off_16_bytes_is_refused(IC):
    """Whichever path the layer runs on."""
    layer = (2, IC, 12, 15, 16, 3, 5, 1, 2)
    batch, _, H, W, OC, kH, kW, stride, pad = layer
    x, w, want = integers(layer)
    lib = load(b16.kernel_library(*LIBS[0]))
    dx, dw = dev(x), dev(w)
    y = torch.full((want.size,), 7.0, dtype=torch.float16, device="cuda:0")
    wsb = lib.conv_workspace_bytes(batch, H, W, IC, OC, kH, kW, stride, pad)
    ws = torch.empty(wsb + 16, dtype=torch.uint8, device="cuda:0")
    rc = lib.conv2d(dx.data_ptr(), dw.data_ptr(), y.data_ptr(), batch, H, W, IC, OC, kH, kW, stride, pad, ws.data_ptr() + 4, wsb,
                    torch.cuda.current_stream().cuda_stream, check=False)
    torch.cuda.synchronize()
    assert rc == HELIX_ERR_INVALID_VALUE and bool((y == 7.0).all())
