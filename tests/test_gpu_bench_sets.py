"""helix_bench_sets and helix_bench_conv_sets: launches that take several sets of operands in turn, in buffers that libraries share."""
import ctypes

import pytest

from utils import hip_ctypes
from utils.helix_runtime import load
from utils.hip_ctypes import HELIX_ERR_INVALID_VALUE, HelixError
from MI355X_FP16 import build_MI355X_FP16 as b16
from MI355X_FP32 import build_MI355X_FP32 as b32

pytestmark = pytest.mark.gpu

LIBRARIES = [b16.kernel_library("gemm", 2, 64, 64, 32, 32, 64), b16.kernel_library("gemv_splitK"), b16.library_for_key(b16.RING_KEYS[0]),
             b32.default_library(), b32.library_for_key(b32.RING_KEYS[0])]


@pytest.mark.parametrize("path", LIBRARIES, ids=lambda p: p.split("/lib")[-1])
def test_times_of_sets_in_turn(path):
    """Sizes off every alignment; a set count is refused before anything is allocated."""
    lib = load(path)
    one = lib.bench(13, 1025, 1032, warmup=2, iters=20)[1]
    turn = lib.bench(13, 1025, 1032, warmup=2, iters=20, sets=3)
    assert turn[0] == turn[1] == turn[2] and 0.3 * one < turn[1] < 10 * one
    with pytest.raises(HelixError) as e:
        lib.bench(13, 1025, 1032, sets=65)
    assert e.value.code == HELIX_ERR_INVALID_VALUE


@pytest.mark.parametrize("path", [LIBRARIES[0], b16.library_for_key(b16.patch_keys()[3]), LIBRARIES[3], b32.library_for_key(b32.patch_keys()[3])],
                         ids=lambda p: p.split("/lib")[-1])
def test_times_of_layers_on_sets_in_turn(path):
    lib, layer = load(path), (3, 16, 19, 17, 40, 3, 3, 1, 1)
    one = lib.bench_conv(*layer, warmup=2, iters=20)[1]
    turn = lib.bench_conv(*layer, warmup=2, iters=20, sets=3)[1]
    assert 0.3 * one < turn < 10 * one
    with pytest.raises(HelixError) as e:
        lib.bench_conv(*layer, sets=65)
    assert e.value.code == HELIX_ERR_INVALID_VALUE


def test_libraries_share_buffers_and_give_them_back():
    """Products and layers, small and larger ones, of two libraries, on one set and on three; a buffer is replaced where it is too small."""
    first, second = load(LIBRARIES[0]), load(LIBRARIES[2])
    with hip_ctypes.shared_buffers():
        buffers = hip_ctypes._buffers.get()
        assert first.bench(256, 512, 640, iters=3, sets=3)[1] > 0
        used = list(buffers.device)
        assert sum(p is not None for p in used) == 10                       # three sets of three, and a workspace
        assert second.bench(256, 520, 648, iters=3, sets=3)[1] > 0 and list(buffers.device) == used
        assert second.bench_conv(2, 16, 9, 9, 24, 3, 3, 1, 1, iters=3, sets=3)[1] > 0 and list(buffers.device) == used
        assert first.bench(256, 512, 640, iters=3)[1] > 0 and first.bench(256, 512, 640, iters=3, rotate_bytes=3 << 20)[1] > 0
        size = buffers.bytes[0]
        assert first.bench(4096, 4096, 1024, iters=3, sets=3)[1] > 0 and buffers.bytes[0] >= 4096 * 1024 * 2 > size
        with pytest.raises(HelixError):
            first.bench(256, 512, 636, iters=3, sets=3)                     # K off 8: refused by the kernel's host side
        assert first.bench(256, 512, 640, iters=3, sets=3)[1] > 0
    assert not any(buffers.device) and not any(buffers.bytes) and hip_ctypes._buffers.get() is None
    assert first._lib.helix_bench_release(ctypes.byref(buffers)) == 0 == first._lib.helix_bench_release(None)
