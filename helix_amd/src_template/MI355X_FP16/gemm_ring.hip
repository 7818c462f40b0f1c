// MI355X (gfx950 / CDNA4) FP16 GEMM and implicit-GEMM convolution template: four waves, K tiles copied straight into a ring of LDS stages.
//
//   C[M x N] = A[M x K] * B[N x K]^T, FP16 in, FP32 accumulate (MFMA), FP16 out; operands and result as in gemm.hip.
//   y[B,OH,OW,OC] = conv2d(x[B,H,W,IC], w[OC,kH,kW,IC]), IC a multiple of 8, at most 31 taps; a 1 x 1 one with stride 1 and no padding
//   is the product of the activations as they lie.
//
// Role in the reference: src_template/Ampere_FP16/gemm.cu:120-534, whose K_STAGE ring of cp.async stages this is the counterpart
// of.
//
// What bounds gemm.hip's tiles on problems of about one round of them is not the matrix pipes but what its waves do beside: eight
// waves read the fragments of a 256 x 192 tile out of LDS with 160 KiB a K tile and write it there with 56, which
// takes 1460 of the 1536 clocks its products need, and tiles are multiples of 32 x 16 with few sizes between.  Here
//   * four waves (two by two, one per SIMD) read 96 KiB for a 224 x 160 tile, and write nothing: every copy is a
//     buffer_load ... lds of 1 KiB (8 rows of 128 bytes), behind its own product;
//   * the ring has K_STAGES stages (three where LDS holds them: the copies of a tile have two tiles to land), one barrier a
//     tile, in the middle of it: each wave has read the tile's second half by then and waited for its copies of the next
//     one, so the barrier both frees the stage and publishes the next;
//   * wave tiles are any multiple of 16 x 16 up to 128 x 128, so that a problem's rows and columns are cut into one round of tiles
//     with little beside them (661 rows into three of 224).
// Measured, us per launch, the fastest of gemm.hip's configurations / of these: 661 x 11008 x 4096 67.1 / 52.4 (224 x 160; 207 tiles on
// 256 CUs, and power: 48 on zeros), 300 x 8192 x 4096 33.2 / 24.7 (160 x 64), 1080 x 6216 x 7760 117 / 102, 611 x 11248 x 3944 69 / 56,
// 1285 x 12144 x 704 30.3 / 26.0, 940 x 1432 x 848 7.9 / 7.0, 3004 x 496 x 464 6.2 / 5.6, 4096 x 3072 x 768 19.9 / 18.8 (128 x 192,
// two stages).  Level or behind: squares from 4096 on (8192^3
// 830 / 855; what both wait for there is L2: 48 KiB a K tile come at 27 - 30 bytes per clock and CU, and the larger tiles that would
// ask for less do not leave room for a third stage), few tiles with long K (split-K libraries).
// Convolutions: a copy's lane knows where the first tap of its pixel lies and which taps are inside the image (a bit each); a tile
// adds the tap's offset, one for all lanes where channels come in 64s.  No table and no register on the way from L2 to LDS, where
// gemm.hip's gather passes staging registers (batch x channels x image, filter; the fastest of gemm.hip and conv_patch.hip / of these):
//   3x3  21 x 384 x 33 x 33 -> 320 58.3 / 48.2   8 x 256 x 75 x 75 -> 512 103 / 93     22 x 192 x 57 x 57 -> 32 21.9 / 19.3
//        32 x 64 x 56 x 56 -> 64 14.7 / 13.6     5 x 64 x 26 x 26 -> 128 5.5 / 4.7     49 x 192 x 22 x 22 -> 64 12.3 / 11.3
// and behind with few tiles and long K, where K is shared out elsewhere (4 x 256 x 14 x 14 7.0 / 9.2); 0.973 in the geometric mean
// over 50 layers.
//
// Compile-time parameters (-D, one shared library per combination):
//   BLOCK_ROWS x BLOCK_COLS   workgroup tile, multiples of 32; a wave's is half of it in both directions
//   K_STAGES                  LDS stages of 64 columns of K
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "helix_abi.h"
#include "helix_fastdiv.h"
#include "helix_ring.h"

#ifndef BLOCK_ROWS
#define BLOCK_ROWS 224
#endif
#ifndef BLOCK_COLS
#define BLOCK_COLS 160
#endif
#ifndef K_STAGES
#define K_STAGES 3
#endif

namespace {

using namespace helix_ring;

typedef _Float16 half_t;
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef int intx2 __attribute__((ext_vector_type(2)));

constexpr int BM = BLOCK_ROWS, BN = BLOCK_COLS, TM = BM / 32, TN = BN / 32, NM = TM * TN, STAGES = K_STAGES, BK = 64;
constexpr int NTHREADS = 256, ROW_BYTES = BK * 2;
constexpr int A_BYTES = BM * ROW_BYTES, STAGE_BYTES = (BM + BN) * ROW_BYTES;
constexpr int COPIES = TM + TN;                     // 1 KiB copies of a wave per K tile
constexpr int STRIP_LD = 32 * TN + 16, STRIP_BYTES = 16 * STRIP_LD;     // results: 16 rows of a wave's columns, rows padded by 16 bytes
constexpr int LDS_BYTES = STAGES * STAGE_BYTES;

static_assert(BM % 32 == 0 && BN % 32 == 0 && TM >= 1 && TN >= 1 && TM <= 8 && TN <= 8, "wave tiles of 16 x 16 .. 128 x 128");
static_assert(STAGES >= 2 && (STAGES - 1) * COPIES <= 63, "copies in flight are counted in a 6-bit counter");
static_assert(LDS_BYTES <= 160 * 1024 && 4 * STRIP_BYTES <= LDS_BYTES, "LDS budget");

struct Params {
    const half_t* A;   // M x K (lda)
    const half_t* B;   // N x K (ldb)
    half_t* C;         // M x N (ldc)
    int M, N, K, lda, ldb, ldc, tiles_m, tiles_n;
};

// A convolution as the implicit GEMM: rows are pixels, columns filters, K the taps' channels
using helix_fastdiv::FastDiv;

struct ConvParams : Params {
    int H, W, IC, kH, kW, stride, pad;
    unsigned x_bytes;
    FastDiv by_OW, by_OH, by_IC, by_kW;
};
constexpr int NO_TAP = 31;                          // a bit that no row's mask has

// What the kernel multiplies: a product, a convolution whose K tiles lie in one tap (channels a multiple of 64), any other
enum { PRODUCT, WHOLE_TAPS, CHUNKS_OF_TAPS };

// (the tile parameters are template arguments for the symbol name's sake: a profiler lists configurations separately)
template <int MODE, class P, int T_STAGES = STAGES, int T_BM = BM, int T_BN = BN>
__global__ __launch_bounds__(NTHREADS, 1) void helix_gemm_f16_ring_kernel(const P p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave >> 1, wave_n = wave & 1, r = lane & 15, q = lane >> 4;

    int tm, tn;
    if (!tile_of((int)blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn)) return;
    const int m0 = tm * BM, n0 = tn * BN;

    // ---- copies: piece d of a wave is 8 LDS rows; row r holds its 16-byte chunk c at c ^ (r / 2 mod 8).  A wave's pieces are all even
    // or all odd, so that a lane has one chunk of every row ------------------------------------------------------------------
    const int rows_a = (p.M - m0) < BM ? (p.M - m0) : BM, rows_b = (p.N - n0) < BN ? (p.N - n0) : BN;
    const half_t* baseA = p.A + (MODE == PRODUCT ? (size_t)m0 * p.lda : 0);
    const half_t* baseB = p.B + (size_t)n0 * p.ldb;
    const unsigned bytesA = (unsigned)(((size_t)(rows_a - 1) * p.lda + p.K) * 2);
    const unsigned bytesB = (unsigned)(((size_t)(rows_b - 1) * p.ldb + p.K) * 2);
    auto piece_of = [&](int d) -> int { return (d < TM ? d : d - TM) * 4 + wave; };
    const int chunk = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7);
    int from[COPIES];
    unsigned inside[TM];                             // of a pixel: the taps that are inside the image; `from` is its first tap's place
#pragma unroll
    for (int d = 0; d < COPIES; d++) {
        const int row = piece_of(d) * 8 + (lane >> 3);
        from[d] = row < (d < TM ? rows_a : rows_b) ? row * (d < TM ? p.lda : p.ldb) * 2 + chunk * 16 : OOB_OFFSET;
        if constexpr (MODE != PRODUCT) {
            if (d >= TM) continue;
            const int m = m0 + row, t = p.by_OW.div(m), ow = m - t * p.by_OW.d, b = p.by_OH.div(t), oh = t - b * p.by_OH.d;
            const int ih = oh * p.stride - p.pad, iw = ow * p.stride - p.pad;
            from[d] = (int)((((unsigned)b * p.H + ih) * p.W + iw) * (unsigned)p.IC * 2u) + (MODE == WHOLE_TAPS ? chunk * 16 : 0);
            const int left = iw < 0 ? -iw : 0, right = p.W - iw < p.kW ? p.W - iw : p.kW;
            const unsigned of_row = right > left ? (1u << right) - (1u << left) : 0u;
            unsigned mask = 0;
            for (int kh = 0; kh < p.kH; kh++) mask |= (unsigned)(ih + kh) < (unsigned)p.H ? of_row << (kh * p.kW) : 0u;
            inside[d] = m < p.M ? mask : 0u;
        }
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)smem;
    // where a product's K is not a multiple of 64 the narrow tile comes first, so that only its copies carry a column mask
    const int ktiles = (p.K + BK - 1) / BK, first_w = MODE == PRODUCT && p.K % BK ? p.K % BK : BK;
    auto k0_of = [&](int t) -> int { return t == 0 ? 0 : first_w + (t - 1) * BK; };
    // a convolution's tap and the byte offset behind a row's first tap, of the tile that is copied next: one for all lanes, or by
    // the lane's chunk
    int tap = 0, offset = 0, kw = 0, c = 0;
    intx4 ra, rb;
    // (past the last tile the copies still go out, from empty buffers: the counts stay)
    auto aim = [&](int t) {
        if constexpr (MODE == PRODUCT) ra = raw_rsrc(baseA + k0_of(t), t < ktiles ? bytesA - (unsigned)k0_of(t) * 2u : 0u);
        else ra = raw_rsrc(p.A, p.x_bytes);
        rb = raw_rsrc(baseB + k0_of(t), t < ktiles ? bytesB - (unsigned)k0_of(t) * 2u : 0u);
        if constexpr (MODE == CHUNKS_OF_TAPS) {
            const int k = t * BK + chunk * 8, at = p.by_IC.div(k), row = p.by_kW.div(at);
            tap = k < p.K ? at : NO_TAP;
            offset = ((row * p.W + at - row * p.kW) * p.IC + k - at * p.IC) * 2;
        }
    };
    auto step = [&]() {                              // to the next tile
        if constexpr (MODE == WHOLE_TAPS) {
            c += BK;
            offset += BK * 2;
            if (c == p.IC) {
                c = 0;
                tap = tap < NO_TAP ? tap + 1 : NO_TAP;
                if (++kw == p.kW) {
                    kw = 0;
                    offset += (p.W - p.kW) * p.IC * 2;
                }
            }
        }
    };
    auto copy = [&](int d, int stage, bool narrow) {
        int at = from[d];
        if (MODE == PRODUCT) at = narrow && chunk * 8 >= first_w ? OOB_OFFSET : at;
        else if (d < TM) at = (inside[d] >> tap) & 1 ? at + offset : OOB_OFFSET;
        else if (MODE == CHUNKS_OF_TAPS) at = tap == NO_TAP ? OOB_OFFSET : at;
        copy16(d < TM ? ra : rb, lds0 + (unsigned)(stage * STAGE_BYTES + (d < TM ? 0 : A_BYTES) + piece_of(d) * 1024), at);
    };
#pragma unroll
    for (int u = 0; u < STAGES; u++) {
        aim(u);
#pragma unroll
        for (int d = 0; d < COPIES; d++) copy(d, u, u == 0);
        step();
    }

    // ---- fragments: lane (r, q) supplies row r, chunk 4 s + q of step s -----------------------------------------------
    int at_a[2], at_b[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const int chunk = ((s * 4 + q) ^ (r >> 1)) << 4;
        at_a[s] = (wave_m * TM * 16 + r) * ROW_BYTES + chunk;
        at_b[s] = A_BYTES + (wave_n * TN * 16 + r) * ROW_BYTES + chunk;
    }
    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    half8 fa[2][TM], fb[2][TN];
    auto read = [&](int e, int s, int stage) {      // in the order in which the products take them: b0, a0 ..., b1 ...
        const unsigned char* base = smem + stage * STAGE_BYTES;
        if (e == 0) fb[s][0] = *(const half8*)(base + at_b[s]);
        else if (e <= TM) fa[s][e - 1] = *(const half8*)(base + at_a[s] + (e - 1) * 16 * ROW_BYTES);
        else fb[s][e - TM] = *(const half8*)(base + at_b[s] + (e - TM) * 16 * ROW_BYTES);
    };
    // the B fragment goes first, which leaves a lane with four consecutive columns of one row
    auto multiply = [&](int g, int s) {
        acc[g % TM][g / TM] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[s][g / TM], fa[s][g % TM], acc[g % TM][g / TM], 0, 0, 0);
    };
    constexpr int EARLY = 2 * NM / 3 > 0 ? 2 * NM / 3 : 1;   // reads end two thirds into a step: the last one arrives before the next

    wait<(STAGES - 1) * COPIES, false>();
    __syncthreads();
#pragma unroll
    for (int e = 0; e < TM + TN; e++) read(e, 0, 0);
    int stage = 0;
    for (int t = 0; t < ktiles; t++) {
        const int next = stage + 1 == STAGES ? 0 : stage + 1;
        aim(t + STAGES);
#pragma unroll
        for (int g = 0; g < NM; g++) {
            multiply(g, 0);
#pragma unroll
            for (int e = 0; e < TM + TN; e++)
                if (e * EARLY / (TM + TN) == g) read(e, 1, stage);
            __builtin_amdgcn_sched_barrier(0);
        }
        // this wave is done reading tile t, and its copies of tile t + 1 have landed; behind the barrier that holds for all
        wait_and_meet<(STAGES - 2) * COPIES>();
#pragma unroll
        for (int g = 0; g < NM; g++) {
            multiply(g, 1);
#pragma unroll
            for (int e = 0; e < TM + TN; e++)
                if (e * EARLY / (TM + TN) == g) read(e, 0, next);    // (past the last tile: zeros, not used)
#pragma unroll
            for (int d = 0; d < COPIES; d++)
                if (d * NM / COPIES == g) copy(d, stage, false);
            __builtin_amdgcn_sched_barrier(0);
        }
        step();
        stage = next;
    }

    // ---- results: 16 rows at a time through LDS, so that a store covers whole pieces of a row --------------------------
    wait<0, true>();
    __syncthreads();                                 // no copy and no read of the ring is left
    unsigned char* strip = smem + wave * STRIP_BYTES;
    // widest store the row stride and base address allow: 8, 4, 2 or 1 halves at a time
    const int align = (int)(((uintptr_t)p.C >> 1) | (unsigned)p.ldc) & 7;
    const int vec = align == 0 ? 8 : (align & 3) == 0 ? 4 : (align & 1) == 0 ? 2 : 1;
    constexpr int CHUNKS = 2 * TN;                   // 16-byte chunks of a strip row
#pragma unroll
    for (int i = 0; i < TM; i++) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const floatx4 a = acc[i][j];
            *(half4*)(strip + r * STRIP_LD + (j * 16 + q * 4) * 2) = half4{(half_t)a[0], (half_t)a[1], (half_t)a[2], (half_t)a[3]};
        }
        __builtin_amdgcn_wave_barrier();             // same-wave LDS traffic stays in program order
#pragma unroll
        for (int u = 0; u < (16 * CHUNKS + 63) / 64; u++) {
            const int idx = u * 64 + lane, row_in = idx / CHUNKS, ch = idx % CHUNKS;
            if (16 * CHUNKS % 64 && row_in >= 16) continue;
            const intx4 v = *(const intx4*)(strip + row_in * STRIP_LD + ch * 16);
            const int row = m0 + (wave_m * TM + i) * 16 + row_in, col = n0 + wave_n * TN * 16 + ch * 8;
            if (row >= p.M || col >= p.N) continue;
            half_t* dst = p.C + (size_t)row * p.ldc + col;
            // non-temporal: the result is not read again by this launch, and the operand panels keep their place in the caches
            if (vec == 8 && col + 8 <= p.N) {
                __builtin_nontemporal_store(v, (intx4*)dst);
            } else if (vec == 4 && col + 8 <= p.N) {
                __builtin_nontemporal_store(intx2{v[0], v[1]}, (intx2*)dst);
                __builtin_nontemporal_store(intx2{v[2], v[3]}, (intx2*)dst + 1);
            } else if (vec == 2 && col + 8 <= p.N) {
#pragma unroll
                for (int e = 0; e < 4; e++) ((int*)dst)[e] = v[e];
            } else {
                const half8 h = __builtin_bit_cast(half8, v);
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (col + e < p.N) dst[e] = h[e];
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

}  // namespace

// -------------------------------------------------------------------------------------------------
// host side
// -------------------------------------------------------------------------------------------------
namespace tpl {

constexpr int kElemBytes = 2;

inline const char* info_json() {
    static char buf[1024];
    static bool done = false;
    if (!done) {
        snprintf(buf, sizeof(buf),
                 "{\"family\": \"gemm_f16\", \"arch\": \"gfx950\", \"mfma\": \"v_mfma_f32_16x16x32_f16\", "
                 "\"k_stages\": %d, \"block_rows\": %d, \"block_cols\": %d, \"wave_rows\": %d, \"wave_cols\": %d, "
                 "\"block_k\": %d, \"split_k\": 1, \"direct_to_lds\": 1, \"threads\": %d, \"lds_bytes\": %d, "
                 "\"layout_a\": \"M x K row-major f16\", \"layout_b\": \"N x K row-major f16\", "
                 "\"layout_c\": \"M x N row-major f16\", \"accumulate\": \"f32\", "
                 "\"k_multiple\": 8, \"ld_multiple\": 8, \"conv\": \"NHWC x [OC][kH][kW][IC]; IC a multiple of 8, at most 31 taps\"}",
                 STAGES, BM, BN, BM / 2, BN / 2, BK, NTHREADS, LDS_BYTES);
        done = true;
    }
    return buf;
}

inline size_t workspace_bytes(int, int, int) { return 0; }
inline size_t conv_workspace_bytes(int, int, int, int, int, int, int, int, int) { return 0; }

inline void bench_layout(int M, int N, int K, size_t* ae, size_t* be, size_t* ce, int* lda, int* ldb, int* ldc) {
    *ae = (size_t)M * K; *be = (size_t)N * K; *ce = (size_t)M * N;
    *lda = K; *ldb = K; *ldc = N;
}

template <int MODE, class P>
inline int launch(const P& p, unsigned grid, hipStream_t s) {
    static int rc = (int)hipFuncSetAttribute((const void*)helix_gemm_f16_ring_kernel<MODE, P>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
    if (rc) return rc;
    hipLaunchKernelGGL((helix_gemm_f16_ring_kernel<MODE, P>), dim3(grid), dim3(NTHREADS), LDS_BYTES, s, p);
    return (int)hipGetLastError();
}

inline int gemm(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc, void*, size_t, hipStream_t s) {
    if (K % 8 != 0 || lda % 8 != 0 || ldb % 8 != 0) return HELIX_ERR_INVALID_VALUE;
    if (lda < K || ldb < K || ldc < N) return HELIX_ERR_INVALID_VALUE;
    if (((uintptr_t)A & 15) || ((uintptr_t)B & 15) || ((uintptr_t)C & 1)) return HELIX_ERR_INVALID_VALUE;
    // per-tile byte offsets are 32-bit
    if ((long long)BM * lda * 2 >= 0x7fffffffLL || (long long)BN * ldb * 2 >= 0x7fffffffLL) return HELIX_ERR_INVALID_VALUE;
    Params p{(const half_t*)A, (const half_t*)B, (half_t*)C, M, N, K, lda, ldb, ldc, (M - 1) / BM + 1, (N - 1) / BN + 1};
    const long long ntiles = (long long)p.tiles_m * p.tiles_n;
    if (ntiles > 0x3fffffffLL) return HELIX_ERR_INVALID_VALUE;
    return launch<PRODUCT>(p, (unsigned)((ntiles + NUM_XCD - 1) / NUM_XCD * NUM_XCD), s);
}

inline int conv2d(const void* x, const void* w, void* y, int batch, int H, int W, int IC, int OC, int kH, int kW, int stride,
                  int pad, void* ws, size_t ws_bytes, hipStream_t s) {
    const int OH = (H + 2 * pad - kH) / stride + 1, OW = (W + 2 * pad - kW) / stride + 1;
    const long long M = (long long)batch * OH * OW, K = (long long)kH * kW * IC, xbytes = (long long)batch * H * W * IC * 2;
    // a 16-byte chunk lies in one tap, and a row's mask has a bit for each and one to spare
    if (IC % 8 != 0 || kH > NO_TAP || kW > NO_TAP || kH * kW > NO_TAP) return HELIX_ERR_UNSUPPORTED;
    if (M > 0x7fffffff || xbytes >= 0x7fffffffLL) return HELIX_ERR_INVALID_VALUE;      // as gemm.hip's
    if (kH == 1 && kW == 1 && stride == 1 && pad == 0) return gemm(x, w, y, (int)M, OC, IC, IC, IC, OC, ws, ws_bytes, s);
    if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)y & 1)) return HELIX_ERR_INVALID_VALUE;
    if (M > 0x7fffffffLL - BM || K > 0x7fffffffLL - 8 * BK || (long long)BN * K * 2 >= 0x7fffffffLL) return HELIX_ERR_INVALID_VALUE;
    ConvParams p;
    static_cast<Params&>(p) = Params{(const half_t*)x, (const half_t*)w, (half_t*)y, (int)M, OC, (int)K, 0, (int)K, OC,
                                     ((int)M - 1) / BM + 1, (OC - 1) / BN + 1};
    p.H = H; p.W = W; p.IC = IC; p.kH = kH; p.kW = kW; p.stride = stride; p.pad = pad;
    p.x_bytes = (unsigned)xbytes;
    p.by_OW = helix_fastdiv::make(OW); p.by_OH = helix_fastdiv::make(OH);
    p.by_IC = helix_fastdiv::make(IC); p.by_kW = helix_fastdiv::make(kW);
    const long long ntiles = (long long)p.tiles_m * p.tiles_n;
    if (ntiles > 0x3fffffffLL) return HELIX_ERR_INVALID_VALUE;
    const unsigned grid = (unsigned)((ntiles + NUM_XCD - 1) / NUM_XCD * NUM_XCD);
    return IC % BK == 0 ? launch<WHOLE_TAPS>(p, grid, s) : launch<CHUNKS_OF_TAPS>(p, grid, s);
}

}  // namespace tpl

#define HELIX_TPL_SCRATCH_BYTES 256   // this family never asks for a workspace
#include "helix_host.h"
