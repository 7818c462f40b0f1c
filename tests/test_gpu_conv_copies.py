"""FP16 convolutions through the workspace: the channel-padded copies and the column buffer of every tile library, and the
layers of one to four channels that the kernel for thin inputs passes on to them -- filters of more than 24 MFMA steps, rows
beyond its LDS, a result off 16 bytes."""
import numpy as np
import pytest
import torch

from utils.helix_runtime import load
from utils.hip_ctypes import HELIX_ERR_INVALID_VALUE
from MI355X_FP16 import build_MI355X_FP16 as b16, MI355X_FP16_conv as c16
from MI355X_FP16 import profile_MI355X_FP16 as p16
from oracle import oracle as O
from gpu_helpers import dev, run_conv

pytestmark = pytest.mark.gpu

KEYS = [k for k in p16.all_keys() if k[0] != 0 and not b16.is_dtl_key(k)]
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


# (batch, IC, H, W, OC, kH, kW, stride, pad)
@pytest.mark.parametrize("layer", [(1, 1, 30, 61, 24, 11, 20, 2, 0),      # 28 MFMA steps: the column buffer ...
                                   (2, 2, 21, 33, 20, 11, 20, 1, 3),
                                   (1, 3, 25, 47, 40, 11, 20, 2, 5),      # ... and the copies
                                   (1, 4, 21, 30, 9, 11, 20, 1, 0),
                                   (60, 1, 9, 3000, 8, 7, 7, 1, 3)],      # an output row's input is beyond LDS
                         ids=lambda l: "x".join(map(str, l)))
def test_layers_the_thin_kernel_refuses(layer):
    assert not c16.runs_thin(*layer)
    x, w, want = integers(layer)
    for cfg in LIBS:
        got = run_conv(load(b16.kernel_library(*cfg)), x, w, layer[7], layer[8], torch.float16)
        assert np.array_equal(got.astype(np.float32), want), cfg


@pytest.mark.parametrize("IC", [1, 2, 3, 4])
def test_result_off_16_bytes(IC):
    """OC a multiple of 8 and y two bytes off: the thin kernel's 16-byte stores do not apply."""
    layer = (2, IC, 12, 15, 16, 3, 5, 1, 2)
    batch, _, H, W, OC, kH, kW, stride, pad = layer
    assert c16.runs_thin(*layer)
    x, w, want = integers(layer)
    for cfg in LIBS:
        lib = load(b16.kernel_library(*cfg))
        dx, dw = dev(x), dev(w)
        y = torch.full((want.size + 9,), 7.0, dtype=torch.float16, device="cuda:0")
        wsb = lib.conv_workspace_bytes(batch, H, W, IC, OC, kH, kW, stride, pad)
        ws = torch.empty(wsb, dtype=torch.uint8, device="cuda:0")
        lib.conv2d(dx.data_ptr(), dw.data_ptr(), y.data_ptr() + 2, batch, H, W, IC, OC, kH, kW, stride, pad, ws.data_ptr(),
                   wsb, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got = y.cpu().numpy().astype(np.float32)
        assert np.array_equal(got[1:1 + want.size].reshape(want.shape), want), cfg
        assert got[0] == 7.0 and (got[1 + want.size:] == 7.0).all(), cfg


@pytest.mark.parametrize("keys", [KEYS[i:i + 60] for i in range(0, len(KEYS), 60)], ids=lambda ks: f"{ks[0]}..")
def test_every_library_copies(keys):
    """Six channels (padded to eight) and one channel with a long filter (column buffer) in every tile library."""
    cases = [(layer, integers(layer)) for layer in ((2, 6, 9, 10, 40, 3, 3, 2, 1), (1, 1, 19, 30, 33, 11, 20, 1, 2))]
    assert not any(c16.runs_thin(*layer) for layer, _ in cases)
    for key in keys:
        lib = load(b16.library_for_key(key))
        for layer, (x, w, want) in cases:
            got = run_conv(lib, x, w, layer[7], layer[8], torch.float16)
            assert np.array_equal(got.astype(np.float32), want), (key, layer)


# pairs of layers on either side of each line of the rule (helix_conv_thin::is_faster)
@pytest.mark.parametrize("layer,thin", [((4, 1, 64, 64, 32, 9, 9, 1, 4), True), ((4, 1, 64, 63, 32, 9, 9, 1, 4), False),
                                        ((2, 2, 64, 64, 72, 11, 11, 1, 5), True), ((2, 2, 64, 63, 72, 11, 11, 1, 5), False),
                                        ((4, 1, 64, 64, 128, 13, 13, 1, 6), True), ((4, 1, 64, 64, 136, 13, 13, 1, 6), False),
                                        ((1, 1, 33, 33, 192, 3, 3, 4, 1), True), ((1, 1, 33, 33, 200, 3, 3, 4, 1), False),
                                        ((1, 4, 33, 33, 448, 1, 1, 4, 0), True), ((1, 4, 33, 33, 456, 1, 1, 4, 0), False),
                                        ((1, 3, 33, 33, 1024, 7, 7, 4, 3), True)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_both_sides_of_the_rule(layer, thin):
    assert c16.runs_thin(*layer) == thin
    x, w, want = integers(layer)
    got = run_conv(load(b16.kernel_library(*LIBS[0])), x, w, layer[7], layer[8], torch.float16)
    assert np.array_equal(got.astype(np.float32), want)


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
