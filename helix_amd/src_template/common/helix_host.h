// Host side shared by every MI355X kernel template: the extern "C" entry points of
// include/helix_abi.h, written once on top of a small per-template interface (namespace tpl).
//
// A template translation unit defines, before including this file:
//   namespace tpl {
//     constexpr int kElemBytes;                       // 2 (FP16) or 4 (FP32)
//     const char* info_json();
//     size_t workspace_bytes(int M, int N, int K);
//     size_t conv_workspace_bytes(int B, int H, int W, int IC, int OC, int kH, int kW, int stride, int pad);
//     int gemm(const void*, const void*, void*, int M, int N, int K, int lda, int ldb, int ldc,
//              void* ws, size_t ws_bytes, hipStream_t);
//     int conv2d(const void*, const void*, void*, int B, int H, int W, int IC, int OC, int kH, int kW,
//                int stride, int pad, void* ws, size_t ws_bytes, hipStream_t);
//     void bench_layout(int M, int N, int K, size_t* a_elems, size_t* b_elems, size_t* c_elems,
//                       int* lda, int* ldb, int* ldc);
//   }
//
// The timing entry points follow the reference's measurement loop (warm-up launches, then a group
// of launches between two events, src_template/Ampere_FP16/gemm.cu:636-652) but initialise their
// buffers, which the reference leaves as returned by cudaMalloc (gemm.cu:630-634).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include <float.h>
#include <vector>

#include "helix_abi.h"

#define HELIX_HIP_TRY(expr)                      \
    do {                                         \
        hipError_t _e = (expr);                  \
        if (_e != hipSuccess) return (int)_e;    \
    } while (0)

namespace helix_host {
namespace {   // internal linkage: a library exports the helix_* entry points only

// Deterministic fill: value = scale * u, u in [-1, 1) from an integer hash of the element index.
__global__ void fill_f16_kernel(_Float16* p, size_t n, float scale, uint32_t seed) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        uint32_t h = (uint32_t)i * 2654435761u + seed;
        h ^= h >> 15; h *= 2246822519u; h ^= h >> 13;
        float u = (float)(h & 0xffffu) * (1.0f / 32768.0f) - 1.0f;
        p[i] = (_Float16)(u * scale);
    }
}

__global__ void fill_f32_kernel(float* p, size_t n, float scale, uint32_t seed) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        uint32_t h = (uint32_t)i * 2654435761u + seed;
        h ^= h >> 15; h *= 2246822519u; h ^= h >> 13;
        float u = (float)(h & 0xffffu) * (1.0f / 32768.0f) - 1.0f;
        p[i] = u * scale;
    }
}

inline int fill(void* p, size_t n_elems, int elem_bytes, float scale, uint32_t seed, hipStream_t s) {
    if (n_elems == 0) return 0;
    int blocks = (int)((n_elems + 255) / 256);
    if (blocks > 4096) blocks = 4096;
    if (elem_bytes == 2)
        hipLaunchKernelGGL(fill_f16_kernel, dim3(blocks), dim3(256), 0, s, (_Float16*)p, n_elems, scale, seed);
    else
        hipLaunchKernelGGL(fill_f32_kernel, dim3(blocks), dim3(256), 0, s, (float*)p, n_elems, scale, seed);
    return (int)hipGetLastError();
}

constexpr size_t kLentUnit = (size_t)2 << 20;    // of lent buffers' sizes, so that the paddings of one problem's layouts fit the same ones

struct DeviceBuffers {
    std::vector<void*> ptrs;
    helix_bench_buffers* lent = nullptr;    // the caller's, taken in order instead of new ones
    int taken = 0;
    ~DeviceBuffers() {
        for (void* p : ptrs)
            if (p) (void)hipFree(p);
    }
    int alloc(void** out, size_t bytes) {
        *out = nullptr;
        if (bytes == 0) bytes = 256;
        if (lent) return take(out, (bytes + kLentUnit - 1) / kLentUnit * kLentUnit);
        hipError_t e = hipMalloc(out, bytes);
        if (e != hipSuccess) {
            (void)hipGetLastError();   // reported here: not by the next launch as well
            return (int)e;
        }
        ptrs.push_back(*out);
        return 0;
    }
    // The next of the caller's buffers, replaced by a larger one where it is too small
    int take(void** out, size_t bytes) {
        if (taken >= HELIX_BENCH_BUFFERS) return HELIX_ERR_INVALID_VALUE;
        void*& p = lent->device[taken];
        size_t& size = lent->bytes[taken];
        if (size < bytes) {
            if (p) (void)hipFree(p);
            size = 0;
            const hipError_t e = hipMalloc(&p, bytes);
            if (e != hipSuccess) {
                (void)hipGetLastError();
                p = nullptr;
                return (int)e;
            }
            size = bytes;
        }
        taken++;
        *out = p;
        return 0;
    }
};

template <typename Launch>
int time_launches(Launch&& launch, hipStream_t s, int warmup, int iters, double* avg_s) {
    if (iters <= 0 || warmup < 0 || !avg_s) return HELIX_ERR_INVALID_VALUE;
    for (int i = 0; i < warmup; i++) {
        int rc = launch(i);
        if (rc) return rc;
    }
    hipEvent_t start, stop;
    HELIX_HIP_TRY(hipEventCreate(&start));
    hipError_t e = hipEventCreate(&stop);
    if (e != hipSuccess) { (void)hipEventDestroy(start); return (int)e; }
    int rc = 0;
    float ms = 0.f;
    e = hipEventRecord(start, s);
    if (e == hipSuccess) {
        for (int i = 0; i < iters && rc == 0; i++) rc = launch(warmup + i);
        if (rc == 0) e = hipEventRecord(stop, s);
        if (rc == 0 && e == hipSuccess) e = hipEventSynchronize(stop);
        if (rc == 0 && e == hipSuccess) e = hipEventElapsedTime(&ms, start, stop);
    }
    (void)hipEventDestroy(start);
    (void)hipEventDestroy(stop);
    if (rc) return rc;
    if (e != hipSuccess) return (int)e;
    *avg_s = (double)ms / 1000.0 / (double)iters;
    return 0;
}

}  // namespace
}  // namespace helix_host

extern "C" {

int helix_info(char* json, int cap) {
    const char* s = tpl::info_json();
    int need = (int)strlen(s) + 1;
    if (json && cap >= need) memcpy(json, s, (size_t)need);
    return need;
}

size_t helix_workspace_bytes(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    return tpl::workspace_bytes(M, N, K);
}

size_t helix_conv_workspace_bytes(int batch, int H, int W, int IC, int OC, int kH, int kW, int stride, int pad) {
    if (batch <= 0 || H <= 0 || W <= 0 || IC <= 0 || OC <= 0 || kH <= 0 || kW <= 0 || stride <= 0 || pad < 0) return 0;
    if (H + 2 * pad < kH || W + 2 * pad < kW) return 0;
    return tpl::conv_workspace_bytes(batch, H, W, IC, OC, kH, kW, stride, pad);
}

int helix_gemm(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc,
               void* workspace, size_t workspace_bytes, void* stream) {
    if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0) return HELIX_ERR_INVALID_VALUE;
    return tpl::gemm(A, B, C, M, N, K, lda, ldb, ldc, workspace, workspace_bytes, (hipStream_t)stream);
}

int helix_conv2d(const void* x, const void* w, void* y, int batch, int H, int W, int IC, int OC, int kH, int kW,
                 int stride, int pad, void* workspace, size_t workspace_bytes, void* stream) {
    if (!x || !w || !y || batch <= 0 || H <= 0 || W <= 0 || IC <= 0 || OC <= 0 || kH <= 0 || kW <= 0 ||
        stride <= 0 || pad < 0)
        return HELIX_ERR_INVALID_VALUE;
    if (H + 2 * pad < kH || W + 2 * pad < kW) return HELIX_ERR_INVALID_VALUE;
    return tpl::conv2d(x, w, y, batch, H, W, IC, OC, kH, kW, stride, pad, workspace, workspace_bytes,
                       (hipStream_t)stream);
}

#ifndef HELIX_NO_STATIC_SCRATCH
}  // extern "C"

// Scratch memory of helix_gemm_static_scratch: the K-partition partial sums live in this array instead of in
// a caller-provided workspace.  Every GPU the library runs on holds its own copy of the array, at its own
// address, until the process ends.  In host code the name is only a handle for HIP_SYMBOL(); the memory is
// reached through the per-device pointer below.
//
// HELIX_TPL_SCRATCH_BYTES (a template may define it before including this file) is the size this library gives the
// array: HELIX_STATIC_SCRATCH_BYTES unless the template never asks for a workspace (tpl::workspace_bytes is 0 for
// every shape), in which case a token array keeps the symbol and the entry point's code path the same.
#ifndef HELIX_TPL_SCRATCH_BYTES
#define HELIX_TPL_SCRATCH_BYTES HELIX_STATIC_SCRATCH_BYTES
#endif
// HELIX_TPL_REQUIRED_BYTES (likewise) names the function that says what a launch of this library must be given:
// tpl::workspace_bytes unless part of that is optional.
#ifndef HELIX_TPL_REQUIRED_BYTES
#define HELIX_TPL_REQUIRED_BYTES tpl::workspace_bytes
#endif
static_assert(HELIX_TPL_SCRATCH_BYTES <= HELIX_STATIC_SCRATCH_BYTES, "the documented maximum bounds every library");
static __device__ __align__(256) unsigned char scratch[HELIX_TPL_SCRATCH_BYTES];

namespace helix_host {
namespace {

constexpr int kMaxDevices = 64;
void* scratch_ptr[kMaxDevices];   // device address of `scratch` per device ordinal, filled on first use

// Device address of `scratch` on the current device (looked up once per device, with that device current).
inline int static_scratch(void** out) {
    int d = -1;
    HELIX_HIP_TRY(hipGetDevice(&d));
    if (d < 0 || d >= kMaxDevices) return HELIX_ERR_INVALID_VALUE;
    void* p = __atomic_load_n(&scratch_ptr[d], __ATOMIC_ACQUIRE);
    if (!p) {
        HELIX_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return HELIX_ERR_INVALID_VALUE;
        __atomic_store_n(&scratch_ptr[d], p, __ATOMIC_RELEASE);   // racing first calls store the same address
    }
    *out = p;
    return 0;
}

}  // namespace
}  // namespace helix_host

extern "C" {

int helix_gemm_static_scratch(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc,
                              void* stream) {
    if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0) return HELIX_ERR_INVALID_VALUE;
    const size_t need = HELIX_TPL_REQUIRED_BYTES(M, N, K);
    if (need > (size_t)HELIX_TPL_SCRATCH_BYTES) return HELIX_ERR_WORKSPACE;
    void* ws = nullptr;
    int rc = helix_host::static_scratch(&ws);
    if (rc) return rc;
    // Nothing to clear: a K-partitioned launch writes every partial sum of its M x N x partitions block before
    // its reduction pass reads that block, and reads nothing else of the array.
    return tpl::gemm(A, B, C, M, N, K, lda, ldb, ldc, ws, (size_t)HELIX_TPL_SCRATCH_BYTES, (hipStream_t)stream);
}
#else
int helix_gemm_static_scratch(const void*, const void*, void*, int, int, int, int, int, int, void*) {
    return HELIX_ERR_UNSUPPORTED;   // vendor comparator: the vendor library manages (and may allocate) its own workspace
}
#endif

int helix_gemm_timed(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc,
                     void* workspace, size_t workspace_bytes, void* stream, int warmup, int iters,
                     double* avg_s) {
    hipStream_t s = (hipStream_t)stream;
    auto launch = [&](int) { return helix_gemm(A, B, C, M, N, K, lda, ldb, ldc, workspace, workspace_bytes, stream); };
    return helix_host::time_launches(launch, s, warmup, iters, avg_s);
}

int helix_conv2d_timed(const void* x, const void* w, void* y, int batch, int H, int W, int IC, int OC, int kH,
                       int kW, int stride, int pad, void* workspace, size_t workspace_bytes, void* stream,
                       int warmup, int iters, double* avg_s) {
    hipStream_t s = (hipStream_t)stream;
    auto launch = [&](int) {
        return helix_conv2d(x, w, y, batch, H, W, IC, OC, kH, kW, stride, pad, workspace, workspace_bytes, stream);
    };
    return helix_host::time_launches(launch, s, warmup, iters, avg_s);
}

}  // extern "C"

namespace helix_host {
namespace {

constexpr int kMaxSets = 64;    // of operands that launches take in turn
static_assert(HELIX_BENCH_BUFFERS >= 3 * kMaxSets + 1, "operands, results and a workspace");

// Mean seconds of `outer` groups of launches: least, mean and largest
template <typename Launch>
int time_groups(Launch&& launch, int warmup, int iters, int outer, double* min_s, double* avg_s, double* max_s) {
    double mn = DBL_MAX, mx = 0.0, tot = 0.0;
    for (int o = 0; o < outer; o++) {
        double t;
        const int rc = time_launches(launch, nullptr, o == 0 ? warmup : 0, iters, &t);
        if (rc) return rc;
        mn = t < mn ? t : mn;
        mx = t > mx ? t : mx;
        tot += t;
    }
    if (min_s) *min_s = mn;
    if (avg_s) *avg_s = tot / outer;
    if (max_s) *max_s = mx;
    return 0;
}

// Allocates and fills one operand `sets` times
inline int alloc_sets(DeviceBuffers& bufs, void* (&out)[kMaxSets], int sets, size_t n_elems, int eb, float scale, uint32_t seed) {
    int rc;
    for (int i = 0; i < sets; i++) {
        if ((rc = bufs.alloc(&out[i], n_elems * eb))) return rc;
        if ((rc = fill(out[i], n_elems, eb, scale, seed + (uint32_t)i, nullptr))) return rc;
    }
    return 0;
}

// `sets` sets of operands and results in turn, of the second operand as many as make `rotate_bytes`
inline int bench_gemm(int M, int N, int K, int warmup, int iters, int outer, int sets, size_t rotate_bytes, helix_bench_buffers* buffers,
                      double* min_s, double* avg_s, double* max_s) {
    size_t ae, be, ce;
    int lda, ldb, ldc;
    tpl::bench_layout(M, N, K, &ae, &be, &ce, &lda, &ldb, &ldc);
    const int eb = tpl::kElemBytes;
    size_t nrot = (size_t)sets;
    if (rotate_bytes > 0 && be * eb > 0) {
        nrot = (rotate_bytes + be * eb - 1) / (be * eb);
        if (nrot < 1) nrot = 1;
        if (nrot > (size_t)kMaxSets) nrot = kMaxSets;
    }
    DeviceBuffers bufs;
    void *As[kMaxSets], *Bs[kMaxSets], *Cs[kMaxSets], *ws;
    const size_t wsb = tpl::workspace_bytes(M, N, K);
    int rc;
    bufs.lent = buffers;
    if ((rc = alloc_sets(bufs, As, sets, ae, eb, 0.5f, 1u))) return rc;
    if ((rc = alloc_sets(bufs, Bs, (int)nrot, be, eb, 0.5f, 2u))) return rc;
    if ((rc = alloc_sets(bufs, Cs, sets, ce, eb, 0.0f, 3u))) return rc;
    if ((rc = bufs.alloc(&ws, wsb))) return rc;
    HELIX_HIP_TRY(hipDeviceSynchronize());

    auto launch = [&](int i) {
        return tpl::gemm(As[(size_t)(i % sets)], Bs[(size_t)i % nrot], Cs[(size_t)(i % sets)], M, N, K, lda, ldb, ldc, ws, wsb, nullptr);
    };
    return time_groups(launch, warmup, iters, outer, min_s, avg_s, max_s);
}

inline int bench_conv(int batch, int IC, int H, int W, int OC, int kH, int kW, int stride, int pad, int warmup, int iters, int outer,
                      int sets, helix_bench_buffers* buffers, double* min_s, double* avg_s, double* max_s) {
    if (batch <= 0 || IC <= 0 || H <= 0 || W <= 0 || OC <= 0 || kH <= 0 || kW <= 0 || stride <= 0 || pad < 0 ||
        iters <= 0 || outer <= 0 || warmup < 0)
        return HELIX_ERR_INVALID_VALUE;
    if (H + 2 * pad < kH || W + 2 * pad < kW) return HELIX_ERR_INVALID_VALUE;
    int OH = (H + 2 * pad - kH) / stride + 1, OW = (W + 2 * pad - kW) / stride + 1;
    size_t xe = (size_t)batch * H * W * IC, we = (size_t)OC * kH * kW * IC, ye = (size_t)batch * OH * OW * OC;
    const int eb = tpl::kElemBytes;
    DeviceBuffers bufs;
    void *xs[kMaxSets], *ws[kMaxSets], *ys[kMaxSets], *scratch;
    const size_t scratch_bytes = tpl::conv_workspace_bytes(batch, H, W, IC, OC, kH, kW, stride, pad);
    int rc;
    bufs.lent = buffers;
    if ((rc = alloc_sets(bufs, xs, sets, xe, eb, 0.5f, 1u))) return rc;
    if ((rc = alloc_sets(bufs, ws, sets, we, eb, 0.5f, 2u))) return rc;
    if ((rc = alloc_sets(bufs, ys, sets, ye, eb, 0.0f, 3u))) return rc;
    if ((rc = bufs.alloc(&scratch, scratch_bytes))) return rc;
    HELIX_HIP_TRY(hipDeviceSynchronize());
    auto launch = [&](int i) {
        return tpl::conv2d(xs[(size_t)(i % sets)], ws[(size_t)(i % sets)], ys[(size_t)(i % sets)], batch, H, W, IC, OC, kH, kW, stride, pad,
                           scratch, scratch_bytes, nullptr);
    };
    return time_groups(launch, warmup, iters, outer, min_s, avg_s, max_s);
}

}  // namespace
}  // namespace helix_host

extern "C" {

int helix_bench(int M, int N, int K, int warmup, int iters, int outer, size_t rotate_bytes, double* min_s,
                double* avg_s, double* max_s) {
    if (M <= 0 || N <= 0 || K <= 0 || iters <= 0 || outer <= 0 || warmup < 0) return HELIX_ERR_INVALID_VALUE;
    return helix_host::bench_gemm(M, N, K, warmup, iters, outer, 1, rotate_bytes, nullptr, min_s, avg_s, max_s);
}

int helix_bench_sets(int M, int N, int K, int warmup, int iters, int sets, size_t rotate_bytes, helix_bench_buffers* buffers, double* avg_s) {
    if (M <= 0 || N <= 0 || K <= 0 || iters <= 0 || warmup < 0 || sets <= 0 || sets > helix_host::kMaxSets) return HELIX_ERR_INVALID_VALUE;
    return helix_host::bench_gemm(M, N, K, warmup, iters, 1, sets, rotate_bytes, buffers, nullptr, avg_s, nullptr);
}

int helix_bench_conv(int batch, int IC, int H, int W, int OC, int kH, int kW, int stride, int pad, int warmup,
                     int iters, int outer, double* min_s, double* avg_s, double* max_s) {
    return helix_host::bench_conv(batch, IC, H, W, OC, kH, kW, stride, pad, warmup, iters, outer, 1, nullptr, min_s, avg_s, max_s);
}

int helix_bench_conv_sets(int batch, int IC, int H, int W, int OC, int kH, int kW, int stride, int pad, int warmup, int iters, int sets,
                          helix_bench_buffers* buffers, double* avg_s) {
    if (sets <= 0 || sets > helix_host::kMaxSets) return HELIX_ERR_INVALID_VALUE;
    return helix_host::bench_conv(batch, IC, H, W, OC, kH, kW, stride, pad, warmup, iters, 1, sets, buffers, nullptr, avg_s, nullptr);
}

int helix_bench_release(helix_bench_buffers* buffers) {
    int rc = 0;
    for (int i = 0; buffers && i < HELIX_BENCH_BUFFERS; i++) {
        const hipError_t e = buffers->device[i] ? hipFree(buffers->device[i]) : hipSuccess;
        if (e != hipSuccess && rc == 0) rc = (int)e;
        buffers->device[i] = nullptr;
        buffers->bytes[i] = 0;
    }
    return rc;
}

}  // extern "C"
