"""The calls this framework's time is measured on: GEMM, decode GEMV and NHWC convolution in FP16 and FP32, each as a
program makes it -- pick the configuration of a problem once (`select_config` over the machine's profile), keep the
library and its workspace, then launch through the library's `gemm` / `conv2d`.

The listed cases and the draws come from the ranges of utils/get_benchmark_shape_list.py: squares, transformer
projections at prefill and decode token counts, GNN feature transforms, CNN layers.  Extents off the tile sizes are
ordinary there (token counts are mostly primes, graphs have any number of nodes), so the draws take any integer.
"""
import math
import os
import sys

import torch

_SCRIPTS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "helix_amd", "scripts")
if os.path.isdir(os.path.join(os.getcwd(), "helix_amd", "scripts")):   # the tree that is run is the working folder's
    _SCRIPTS = os.path.join(os.getcwd(), "helix_amd", "scripts")
if _SCRIPTS not in sys.path:
    sys.path.insert(0, _SCRIPTS)

LARGEST_FLOPS = 2.0 * 8192 ** 3      # FP16; draws stay below the largest listed case
LARGEST_BYTES = 600e6
LARGEST_FLOPS_F32 = 6e10


def _gemm(name, dtype, M, N, K, kind="gemm"):
    return {"name": name, "op": kind, "dtype": dtype, "M": M, "N": N, "K": K}


def _conv(name, dtype, batch, IC, H, W, OC, kH, kW, stride, pad):
    return {"name": name, "op": "conv", "dtype": dtype, "batch": batch, "IC": IC, "H": H, "W": W, "OC": OC, "kH": kH,
            "kW": kW, "stride": stride, "pad": pad}


def listed():
    return [
        # one decode step of one sequence through a 4096-wide projection: the smallest call, launch and latency count
        _gemm("decode_f16_m1", "f16", 1, 4096, 4096, "decode"),
        # sixteen sequences in decode through the largest weight matrix of the decode list
        _gemm("decode_f16_m16", "f16", 16, 28672, 8192, "decode"),
        # the same at full precision: four sequences, LLaMA-2's up projection
        _gemm("decode_f32_m4", "f32", 4, 11008, 4096, "decode"),
        # prefill of one prompt of 661 tokens (a prime: rows off every tile) through LLaMA-2's up projection
        _gemm("prefill_f16_661", "f16", 661, 11008, 4096),
        # a BERT-base FFN projection at batch 8, sequence 512: one of the ordinary mid-size products
        _gemm("bert_f16_ffn", "f16", 4096, 3072, 768),
        # the large square, the headline product
        _gemm("square_f16_8192", "f16", 8192, 8192, 8192),
        # first feature transform of a two-layer GCN (334863 nodes, 96 features, 16 hidden): tall and skinny
        _gemm("gnn_f16", "f16", 334863, 16, 96),
        # FP32, every extent off the tiles
        _gemm("irregular_f32", "f32", 4000, 2300, 770),
        # first layer of ResNet / GoogleNet at batch 32: three channels, stride 2
        _conv("conv_f16_first", "f16", 32, 3, 224, 224, 64, 7, 7, 2, 3),
        # first residual stage at batch 32: large image, few channels
        _conv("conv_f16_56x56x64", "f16", 32, 64, 56, 56, 64, 3, 3, 1, 1),
        # third residual stage at batch 4 (an inference batch): small image, more channels, few output tiles
        _conv("conv_f16_14x14x256", "f16", 4, 256, 14, 14, 256, 3, 3, 1, 1),
        # second residual stage at batch 32 in FP32
        _conv("conv_f32_28x28x128", "f32", 32, 128, 28, 28, 128, 3, 3, 1, 1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        flops = LARGEST_FLOPS if case["dtype"] == "f16" else LARGEST_FLOPS_F32
        if w["flops"] <= flops and w["bytes"] <= LARGEST_BYTES and max(w["bytes"], w["flops"] / 300.0) >= 2e6:
            return {k: v for k, v in case.items() if k != "name"}


def _draw(rng):
    what = rng.choice(("decode", "decode", "prefill", "prefill", "prefill", "gnn", "conv", "conv", "conv", "first"))
    dtype = "f16" if rng.random() < 0.7 else "f32"
    # projections' widths are mostly multiples of 8, the rest of the range is any integer
    width = (lambda lo, hi: _log_int(rng, lo / 8, hi / 8) * 8) if rng.random() < 0.7 else (lambda lo, hi: _log_int(rng, lo, hi))
    if what == "decode":
        return _gemm("", dtype, rng.randint(1, 16), width(1024, 28672), width(1024, 13824), "decode")
    if what == "prefill":
        return _gemm("", dtype, _log_int(rng, 17, 8192), width(256, 15360), width(256, 13824))
    if what == "gnn":
        return _gemm("", dtype, _log_int(rng, 20000, 1900000), _log_int(rng, 2, 128), _log_int(rng, 16, 1400))
    batch = _log_int(rng, 1, 64)
    if what == "first":
        k = rng.choice((3, 5, 7, 11))
        side = rng.randint(100, 224)
        return _conv("", dtype, batch, 3, side, side, rng.choice((32, 48, 64, 96)), k, k, rng.choice((1, 2, 4)), k // 2)
    k = rng.choice((1, 1, 3, 3, 3, 5))
    side = _log_int(rng, 7, 112)
    ic = rng.choice((16, 24, 25, 32, 48, 64, 96, 112, 128, 144, 192, 256, 384, 480, 512, 832))
    oc = rng.choice((16, 32, 48, 64, 96, 128, 160, 192, 208, 256, 320, 384, 512))
    return _conv("", dtype, batch, ic, side, side, oc, k, k, 2 if k > 1 and rng.random() < 0.2 else 1, k // 2)


def _out_extents(case):
    OH = (case["H"] + 2 * case["pad"] - case["kH"]) // case["stride"] + 1
    OW = (case["W"] + 2 * case["pad"] - case["kW"]) // case["stride"] + 1
    return OH, OW


def work(case):
    eb = 2 if case["dtype"] == "f16" else 4
    if case["op"] == "conv":
        OH, OW = _out_extents(case)
        weights = case["OC"] * case["kH"] * case["kW"] * case["IC"]
        pixels = case["batch"] * OH * OW
        return {"bytes": float(eb * (case["batch"] * case["H"] * case["W"] * case["IC"] + weights + pixels * case["OC"])),
                "flops": 2.0 * pixels * weights}
    M, N, K = case["M"], case["N"], case["K"]
    return {"bytes": float(eb * (M * K + N * K + M * N)), "flops": 2.0 * M * N * K}


def tolerance(case):
    """FP16 results: the rounding of the result over FP32 sums, 2.1e-4 in the norm and 4.9e-4 at most against the same
    product in 64 bits.  FP32: sums of K products in another order; against 64 bits 5e-7 in the norm (4e-6 at most) at
    K = 770, 6e-7 (5e-6) at K = 1152, growing with the root of K to about four times that at the longest K drawn."""
    return {"rel": 8e-4, "max": 2e-3} if case["dtype"] == "f16" else {"rel": 8e-6, "max": 8e-5}


_profiles = {}


def _profile(backend):
    """The machine's profile of a backend: read from build/prof_dict, made there once (seconds) if it is missing."""
    if backend not in _profiles:
        import importlib
        from utils.helix_runtime import prof_dict_path, read_prof_dict
        if not os.path.exists(prof_dict_path(backend)):
            getattr(importlib.import_module(f"{backend}.profile_{backend}"), f"profile_Helix_{backend}_gemm_kernel")()
        _profiles[backend] = read_prof_dict(backend)
    return _profiles[backend]


def _modules(dtype):
    if dtype == "f16":
        from MI355X_FP16 import MI355X_FP16_conv as conv, MI355X_FP16_gemm as gemm, build_MI355X_FP16 as build
        return "MI355X_FP16", gemm, conv, build, torch.float16
    from MI355X_FP32 import MI355X_FP32_conv as conv, MI355X_FP32_gemm as gemm, build_MI355X_FP32 as build
    return "MI355X_FP32", gemm, conv, build, torch.float32


def prepare(case, seed):
    from utils.helix_runtime import load
    backend, gemm, conv, build, dtype = _modules(case["dtype"])
    prof = _profile(backend)
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(int(seed))

    def normal(shape, std):
        return torch.randn(shape, generator=gen, device=dev, dtype=torch.float32).mul_(std).to(dtype)

    if case["op"] == "conv":
        layer = tuple(case[k] for k in ("batch", "IC", "H", "W", "OC", "kH", "kW", "stride", "pad"))
        batch, IC, H, W, OC, kH, kW, stride, pad = layer
        lib = load(build.library_for_key(conv.select_config(prof, *layer)))
        OH, OW = _out_extents(case)
        x = normal((batch, H, W, IC), 0.05)
        w = normal((OC, kH, kW, IC), 0.05)
        y = torch.empty((batch, OH, OW, OC), dtype=dtype, device=dev)
        ws_bytes = lib.conv_workspace_bytes(batch, H, W, IC, OC, kH, kW, stride, pad)
        ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=dev)
        return {"launch": lib.conv2d, "keep": (x, w, ws), "out": y, "transposed": None,
                "args": (x.data_ptr(), w.data_ptr(), y.data_ptr(), batch, H, W, IC, OC, kH, kW, stride, pad,
                         ws.data_ptr(), ws_bytes, torch.cuda.current_stream().cuda_stream)}

    M, N, K = case["M"], case["N"], case["K"]
    a_std, b_std = (1.0, 0.02) if case["op"] == "decode" else (0.1, 0.1)
    A = normal((M, K), a_std)
    B = normal((N, K), b_std)          # weights as the framework stores them: one row per output column
    key = gemm.select_config(prof, M, N, K)
    lib = load(build.library_for_key(key))
    out = torch.empty((M, N), dtype=dtype, device=dev)
    transposed = None
    if lib.info()["family"] == "sgemm_f32":     # both operands K-major, rows of whole 16-byte chunks
        A, B = _padded(A.t(), 4), _padded(B.t(), 4)
        m, n, k, lda, ldb, C = M, N, K, A.shape[1], B.shape[1], out
    else:
        step = 8 if case["dtype"] == "f16" else 4
        A, B = _padded(A, step), _padded(B, step)
        k = A.shape[1]
        m, n, lda, ldb, C = M, N, k, k, out
        if lib.info()["family"].startswith("gemv") and M > N:     # it streams its second operand: C^T = B A^T
            A, B, m, n = B, A, N, M
            C = transposed = torch.empty((N, M), dtype=dtype, device=dev)
    ws_bytes = lib.workspace_bytes(m, n, k)
    ws = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=dev)
    return {"launch": lib.gemm, "keep": (A, B, ws), "out": out, "transposed": transposed,
            "args": (A.data_ptr(), B.data_ptr(), C.data_ptr(), m, n, k, lda, ldb, n, ws.data_ptr(), ws_bytes,
                     torch.cuda.current_stream().cuda_stream)}


def _padded(t, step):
    """Contiguous, columns zero-padded to a multiple of `step`."""
    cols = -(-t.shape[1] // step) * step
    if cols == t.shape[1]:
        return t.contiguous()
    p = torch.zeros((t.shape[0], cols), dtype=t.dtype, device=t.device)
    p[:, :t.shape[1]] = t
    return p


def run(state):
    state["launch"](*state["args"])
    if state["transposed"] is not None:
        state["out"].copy_(state["transposed"].t())
    return state["out"]
