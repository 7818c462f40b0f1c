// MI355X (gfx950 / CDNA4) FP32 GEMM template: four waves, K tiles copied straight into a ring of LDS stages.
//
//   C[M x N] = A^T * B with A stored K x M and B stored K x N (row-major FP32): operands and result as in sgemm.hip.
//
// Role in the reference: src_template/Ampere_FP32/sgemm.cu:97-350, whose cp.async stages this is the counterpart of.
//
// Bound: the matrix pipes (256 flop per clock and CU: 157 TFLOP/s).  What sgemm.hip's tiles lose beside the products is issue slots:
// a K tile passes through staging registers into LDS, and its fragments come as scalars.  Here
//   * copies are buffer_load ... lds of 1 KiB, issued behind the products; both operands lie K-major, so that a stage is 32 rows of
//     BLOCK_ROWS and BLOCK_COLS floats as they are in memory, and rows from K on are beyond the buffer, hence zeros;
//   * v_mfma_f32_16x16x4_f32 takes one float of a row per lane; it does not matter which row of the wave's tile is lane r's, so
//     a lane reads four consecutive rows of a k in 16 bytes, one for each of four tiles, and holds four consecutive columns of a result
//     row in return, which it stores in 16 bytes, a quarter wave 256 bytes together.  The loop for a 96 x 96 wave tile: 288 products,
//     32 LDS reads, 12 copies, 3 waits, one barrier per 32 columns of K;
//   * tiles are any multiple of 32 x 32, and the last half K tile is left out where it is empty (K = 770: 784 columns of work).
// Two stages do (a K tile of the smallest workgroup takes 1000 clocks), which leaves room for up to eight workgroups on a CU: one's
// stores and first copies lie behind another's products.
// Sums: ascending k, one FMA chain per result, as sgemm.hip's unpartitioned launches; the same bits in every configuration over
// 300 x 520 x 100, 1000 x 770 x 777 and 513 x 257 x 16.
// Measured, us per launch, the fastest of sgemm.hip's configurations / of these: 4000 x 2300 x 770 120.7 / 107.2 (64 x 64 tiles; 94 are
// the products at the peak rate), 2048^3 129.9 / 121.4, 4096^3 946 / 925, 661 x 11008 x 1024 128.8 / 116.5, 512 x 3072 x 768 25.7 / 22.6,
// 8134 x 451 x 5225 326 / 293, 283256 x 72 x 331 196 / 168, 3325 x 1824 x 328 37.5 / 33.1, 196 x 512 x 256 5.4 / 4.6.  Behind where
// tiles are few and K is long (29 x 1000 x 11976 18.8 / 105): K groups and partitions stay sgemm.hip's, as do convolutions.
//
// Compile-time parameters (-D, one shared library per combination):
//   BLOCK_ROWS x BLOCK_COLS   workgroup tile, multiples of 32; a wave's is half of it in both directions
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <utility>

#include "helix_abi.h"
#include "helix_ring.h"

#ifndef BLOCK_ROWS
#define BLOCK_ROWS 192
#endif
#ifndef BLOCK_COLS
#define BLOCK_COLS 192
#endif

namespace {

using namespace helix_ring;

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int BM = BLOCK_ROWS, BN = BLOCK_COLS, TM = BM / 32, TN = BN / 32, NM = TM * TN, STAGES = 2, BK = 32;
constexpr int NTHREADS = 256, STEPS = BK / 8;       // k steps of four in half a K tile
constexpr int A_BYTES = BM * BK * 4, STAGE_BYTES = (BM + BN) * BK * 4, LDS_BYTES = STAGES * STAGE_BYTES;
constexpr int COPIES = TM + TN;                     // 1 KiB copies of a wave per K tile

static_assert(BM % 32 == 0 && BN % 32 == 0 && TM >= 1 && TN >= 1 && TM <= 8 && TN <= 8, "wave tiles of 16 x 16 .. 128 x 128");
static_assert((STAGES - 1) * COPIES <= 63, "copies in flight are counted in a 6-bit counter");
static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");

// A wave's T tiles of 16 rows (or columns) lie in groups of 4, 2 and 1: lane r of a group of W holds its W r .. W r + W - 1, in one
// load or store of W floats, so tile i of the group is made of every W-th row.
constexpr int groups(int T) { return T / 4 + (T >> 1 & 1) + (T & 1); }
constexpr int group_first(int T, int g) { return g < T / 4 ? 4 * g : g == T / 4 && (T & 2) ? T / 4 * 4 : T - 1; }
constexpr int group_width(int T, int g) { return g < T / 4 ? 4 : g == T / 4 && (T & 2) ? 2 : 1; }
constexpr int group_of(int T, int t) { return t < T / 4 * 4 ? t / 4 : (T & 2) && t < T / 4 * 4 + 2 ? T / 4 : groups(T) - 1; }
constexpr int GA = groups(TM), GB = groups(TN);

struct Params {
    const float* A;    // K x M (lda)
    const float* B;    // K x N (ldb)
    float* C;          // M x N (ldc)
    int M, N, K, lda, ldb, ldc, tiles_m, tiles_n;
};

// f(0) .. f(N - 1) with constant arguments: the K loop's several hundred steps are more than `#pragma unroll` takes in nested loops
template <int N, class F, int... I>
__device__ __forceinline__ void each(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void each(F&& f) {
    each<N>(f, std::make_integer_sequence<int, N>{});
}

template <int W>
__device__ __forceinline__ void load(const unsigned char* from, float* to) {
    if (W == 4) {
        const floatx4 v = *(const floatx4*)from;
        to[0] = v[0]; to[1] = v[1]; to[2] = v[2]; to[3] = v[3];
    } else if (W == 2) {
        const floatx2 v = *(const floatx2*)from;
        to[0] = v[0]; to[1] = v[1];
    } else {
        to[0] = *(const float*)from;
    }
}

// (the tile parameters are template arguments for the symbol name's sake: a profiler lists configurations separately)
template <int T_BM = BM, int T_BN = BN>
__global__ __launch_bounds__(NTHREADS, 1) void helix_sgemm_f32_ring_kernel(const Params p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave >> 1, wave_n = wave & 1, r = lane & 15, q = lane >> 4;
    int tm, tn;
    if (!tile_of((int)blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn)) return;
    const int m0 = tm * BM, n0 = tn * BN;

    // ---- copies: a stage holds 32 rows of A's BM columns, then of B's BN; a wave's piece is 64 chunks of 16 bytes of them -----
    // (whole rows of lda and ldb are inside the buffers, rows from K on are not; columns beyond M and N that lie in a chunk of the
    // last ones go into results that are not stored)
    int from[COPIES];
#pragma unroll
    for (int d = 0; d < COPIES; d++) {
        const int T = d < TM ? BM : BN, chunk = (d < TM ? wave * TM + d : wave * TN + d - TM) * 64 + lane;
        const int row = chunk / (T / 4), col = chunk % (T / 4) * 4;
        from[d] = (d < TM ? m0 : n0) + col < (d < TM ? p.M : p.N) ? (row * (d < TM ? p.lda : p.ldb) + col) * 4 : OOB_OFFSET;
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)smem;
    const int ktiles = (p.K + BK - 1) / BK;
    // (past the last tile the copies still go out, from empty buffers: the counts stay)
    auto rsrc_of = [&](const float* base, int ld, int first, int t) -> intx4 {
        const int k0 = t < ktiles ? t * BK : 0;
        return raw_rsrc(base + (size_t)k0 * ld + first, t < ktiles ? (unsigned)(((size_t)(p.K - k0) * ld - first) * 4) : 0u);
    };
    auto copy = [&](int d, int stage, const intx4& ra, const intx4& rb) {
        const int piece = d < TM ? wave * TM + d : wave * TN + d - TM;
        copy16(d < TM ? ra : rb, lds0 + (unsigned)(stage * STAGE_BYTES + (d < TM ? 0 : A_BYTES) + piece * 1024), from[d]);
    };
#pragma unroll
    for (int u = 0; u < STAGES; u++) {
        const intx4 ra = rsrc_of(p.A, p.lda, m0, u), rb = rsrc_of(p.B, p.ldb, n0, u);
#pragma unroll
        for (int d = 0; d < COPIES; d++) copy(d, u, ra, rb);
    }

    // ---- fragments: lane (r, q) supplies row k = 4 step + q; see group_first --------------------------------------------
    int at_a[GA], at_b[GB];
#pragma unroll
    for (int g = 0; g < GA; g++) at_a[g] = (q * BM + (wave_m * TM + group_first(TM, g)) * 16 + group_width(TM, g) * r) * 4;
#pragma unroll
    for (int g = 0; g < GB; g++) at_b[g] = A_BYTES + (q * BN + (wave_n * TN + group_first(TN, g)) * 16 + group_width(TN, g) * r) * 4;
    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    float fa[2][STEPS][TM], fb[2][STEPS][TN];
    constexpr int READS = STEPS * (GA + GB);
    auto read = [&](int e, int h, int stage) {       // step by step, in the order in which the products take them
        const unsigned char* base = smem + stage * STAGE_BYTES;
        const int s = e / (GA + GB), g = e % (GA + GB);
        if (g < GA) {
            const unsigned char* src = base + at_a[g] + (h * STEPS + s) * 4 * BM * 4;
            float* dst = &fa[h][s][group_first(TM, g)];
            if (group_width(TM, g) == 4) load<4>(src, dst);
            else if (group_width(TM, g) == 2) load<2>(src, dst);
            else load<1>(src, dst);
        } else {
            const unsigned char* src = base + at_b[g - GA] + (h * STEPS + s) * 4 * BN * 4;
            float* dst = &fb[h][s][group_first(TN, g - GA)];
            if (group_width(TN, g - GA) == 4) load<4>(src, dst);
            else if (group_width(TN, g - GA) == 2) load<2>(src, dst);
            else load<1>(src, dst);
        }
    };
    constexpr int PRODUCTS = STEPS * NM;
    auto multiply = [&](int g, int h) {
        const int s = g / NM, i = g % NM % TM, j = g % NM / TM;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[h][s][i], fb[h][s][j], acc[i][j], 0, 0, 0);
    };
    // fragment reads that are out after g products: they end two thirds into a half
    auto due = [](int g, int reads) constexpr -> int { return 3 * g >= 2 * PRODUCTS ? reads : 3 * g * reads / (2 * PRODUCTS); };

    wait<(STAGES - 1) * COPIES, false>();
    __syncthreads();
    each<READS>([&](auto e) __attribute__((always_inline)) { read(e, 0, 0); });
    int stage = 0;
    // (whole tiles, and half a one behind the loop where no more is left: a way out in the middle of the loop had the compiler copy
    // every accumulator twice a tile)
    const int halves = (p.K + BK / 2 - 1) / (BK / 2);
    for (int t = 0; t < halves / 2; t++) {
        const int next = stage + 1 == STAGES ? 0 : stage + 1;
        const intx4 ra = rsrc_of(p.A, p.lda, m0, t + STAGES), rb = rsrc_of(p.B, p.ldb, n0, t + STAGES);
        each<PRODUCTS>([&](auto g) __attribute__((always_inline)) {
            multiply(g, 0);
#pragma unroll
            for (int e = due(g, READS); e < due(g + 1, READS); e++) read(e, 1, stage);
            __builtin_amdgcn_sched_barrier(0);
        });
        // this wave is done reading tile t, and its copies of tile t + 1 have landed; behind the barrier that holds for all
        wait_and_meet<(STAGES - 2) * COPIES>();
        each<PRODUCTS>([&](auto g) __attribute__((always_inline)) {
            multiply(g, 1);
#pragma unroll
            for (int e = due(g, READS); e < due(g + 1, READS); e++) read(e, 0, next);   // (past the last tile: zeros, not used)
#pragma unroll
            for (int d = g * COPIES / PRODUCTS; d < (g + 1) * COPIES / PRODUCTS; d++) copy(d, stage, ra, rb);
            __builtin_amdgcn_sched_barrier(0);
        });
        stage = next;
    }
    if (halves & 1) each<PRODUCTS>([&](auto g) __attribute__((always_inline)) { multiply(g, 0); });
    wait<0, true>();                                 // no copy is left when the workgroup gives its LDS back

    // ---- results: lanes 0 .. 15 of a quarter hold a piece of a row, 256, 128 or 64 bytes long -----------------------------
    const int align = (int)(((uintptr_t)p.C >> 2) | (unsigned)p.ldc) & 3;
    const int vec = align == 0 ? 4 : align == 2 ? 2 : 1;     // widest store the row stride and base address allow
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int ga = group_of(TM, i), first = group_first(TM, ga), width = group_width(TM, ga);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = m0 + (wave_m * TM + first) * 16 + width * (4 * q + v) + i - first;
            if (row >= p.M) continue;
#pragma unroll
            for (int g = 0; g < GB; g++) {
                const int j = group_first(TN, g), w = group_width(TN, g);
                const int col = n0 + (wave_n * TN + j) * 16 + w * r;
                float* dst = p.C + (size_t)row * p.ldc + col;
                if (w == 4 && vec == 4 && col + 4 <= p.N) {
                    __builtin_nontemporal_store(floatx4{acc[i][j][v], acc[i][j + w / 4][v], acc[i][j + w / 2][v], acc[i][j + w - 1][v]},
                                                (floatx4*)dst);
                } else if (w >= 2 && vec >= 2 && col + w <= p.N) {
#pragma unroll
                    for (int e = 0; e < w; e += 2)
                        __builtin_nontemporal_store(floatx2{acc[i][j + e][v], acc[i][j + e + 1][v]}, (floatx2*)(dst + e));
                } else {
#pragma unroll
                    for (int e = 0; e < w; e++)
                        if (col + e < p.N) dst[e] = acc[i][j + e][v];
                }
            }
        }
    }
}

}  // namespace

// -------------------------------------------------------------------------------------------------
// host side
// -------------------------------------------------------------------------------------------------
namespace tpl {

constexpr int kElemBytes = 4;

inline const char* info_json() {
    static char buf[1024];
    static bool done = false;
    if (!done) {
        snprintf(buf, sizeof(buf),
                 "{\"family\": \"sgemm_f32\", \"arch\": \"gfx950\", \"mfma\": \"v_mfma_f32_16x16x4_f32\", "
                 "\"k_stages\": %d, \"block_rows\": %d, \"block_cols\": %d, \"wave_rows\": %d, \"wave_cols\": %d, "
                 "\"block_k\": %d, \"k_groups\": 1, \"split_k\": 1, \"direct_to_lds\": 1, \"threads\": %d, \"lds_bytes\": %d, "
                 "\"layout_a\": \"K x M row-major f32\", \"layout_b\": \"K x N row-major f32\", "
                 "\"layout_c\": \"M x N row-major f32\", \"accumulate\": \"f32\", "
                 "\"k_multiple\": 1, \"ld_multiple\": 4, \"conv\": \"none\"}",
                 STAGES, BM, BN, BM / 2, BN / 2, BK, NTHREADS, LDS_BYTES);
        done = true;
    }
    return buf;
}

inline size_t workspace_bytes(int, int, int) { return 0; }
inline size_t conv_workspace_bytes(int, int, int, int, int, int, int, int, int) { return 0; }

inline void bench_layout(int M, int N, int K, size_t* ae, size_t* be, size_t* ce, int* lda, int* ldb, int* ldc) {
    const int Mp = (M + 3) / 4 * 4, Np = (N + 3) / 4 * 4;
    *ae = (size_t)K * Mp; *be = (size_t)K * Np; *ce = (size_t)M * Np;
    *lda = Mp; *ldb = Np; *ldc = Np;
}

inline int gemm(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc, void*, size_t, hipStream_t s) {
    if (lda % 4 != 0 || ldb % 4 != 0) return HELIX_ERR_INVALID_VALUE;  // 16-byte copies along M and N
    if (lda < M || ldb < N || ldc < N) return HELIX_ERR_INVALID_VALUE;
    if (((uintptr_t)A & 15) || ((uintptr_t)B & 15) || ((uintptr_t)C & 3)) return HELIX_ERR_INVALID_VALUE;
    // byte offsets inside one K tile are 32-bit, and a buffer descriptor spans at most 4 GiB
    if ((long long)K * lda * 4 >= 0xffffffffLL || (long long)K * ldb * 4 >= 0xffffffffLL) return HELIX_ERR_INVALID_VALUE;
    if ((long long)BK * lda * 4 >= 0x7fffffffLL || (long long)BK * ldb * 4 >= 0x7fffffffLL) return HELIX_ERR_INVALID_VALUE;
    Params p{(const float*)A, (const float*)B, (float*)C, M, N, K, lda, ldb, ldc, (M - 1) / BM + 1, (N - 1) / BN + 1};
    const long long ntiles = (long long)p.tiles_m * p.tiles_n;
    if (ntiles > 0x3fffffffLL) return HELIX_ERR_INVALID_VALUE;
    static int rc = (int)hipFuncSetAttribute((const void*)helix_sgemm_f32_ring_kernel<>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
    if (rc) return rc;
    const unsigned grid = (unsigned)((ntiles + NUM_XCD - 1) / NUM_XCD * NUM_XCD);
    hipLaunchKernelGGL(helix_sgemm_f32_ring_kernel<>, dim3(grid), dim3(NTHREADS), LDS_BYTES, s, p);
    return (int)hipGetLastError();
}

inline int conv2d(const void*, const void*, void*, int, int, int, int, int, int, int, int, int, void*, size_t, hipStream_t) {
    return HELIX_ERR_UNSUPPORTED;
}

}  // namespace tpl

#define HELIX_TPL_SCRATCH_BYTES 256   // this family never asks for a workspace
#include "helix_host.h"
