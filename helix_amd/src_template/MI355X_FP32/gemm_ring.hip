// MI355X (gfx950 / CDNA4) FP32 GEMM and implicit-GEMM convolution template: four waves, K tiles copied straight into a ring of LDS stages.
//
//   C[M x N] = A^T * B with A stored K x M and B stored K x N (row-major FP32): operands and result as in sgemm.hip.
//   y[B,OH,OW,OC] = conv2d(x[B,H,W,IC], w[OC,kH,kW,IC]), IC a multiple of 4, at most 31 taps.
//
// Role in the reference: src_template/Ampere_FP32/sgemm.cu:97-350, whose cp.async stages this is the counterpart of.
//
// Bound: the matrix pipes (256 flop per clock and CU: 157 TFLOP/s).  What sgemm.hip's tiles lose beside the products is issue slots:
// a K tile passes through staging registers into LDS, and its fragments come as scalars.  Here
//   * copies are buffer_load ... lds of 1 KiB, issued behind the products; both operands lie K-major, so that a stage is 32 rows of
//     BLOCK_ROWS and BLOCK_COLS floats as they are in memory, and rows from K on are beyond the buffer, hence zeros;
//   * v_mfma_f32_16x16x4_f32 takes one float of a row per lane; it does not matter which row of the wave's tile is lane r's, so
//     a lane reads four consecutive rows of a k in 16 bytes, one for each of four tiles, and holds four consecutive columns of a result
//     row in return, which it stores in 16 bytes, a quarter wave 256 bytes together.  The loop for a 64 x 64 wave tile (64 x 256
//     in all): 128 products, 16 LDS reads, 10 copies, one barrier per 32 columns of K;
//   * the four waves lie 2 x 2, or in a row or column, which gives tiles 16 rows or columns apart: 48 and 80 columns for products
//     and layers of few; and the last half K tile is left out where it is empty (K = 770: 784 columns of work).
// Two stages do (the products of a K tile take 256 clocks a wave at the least), which leaves room for up to eight workgroups on a CU: one's
// stores and first copies lie behind another's products.
// Sums (common/helix_sums.h): ascending k, of many results a chain of FMAs per 256 of K, added in order: up to there the bits of an
// unpartitioned sgemm.hip launch.  2.9e-7 - 3.0e-7 in the norm from K = 770 to 6160, where one chain leaves 5.0e-7 - 14e-7, sgemm.hip's
// two K groups 3.5e-7 - 9.9e-7 and its partitions 3.9e-7 - 13e-7 (operands ~ N(0, 1)).  Of few results a chain per 16, as exact as sgemm.hip's
// four and eight K groups: 1.1e-7 - 1.5e-7 from K = 256 to 776.
// Measured, us per launch, the fastest of sgemm.hip's configurations / of these: 4000 x 2300 x 770 119.3 / 109.4 (94 are the products
// at the peak rate), 2048^3 130.0 / 123.5, 4096^3 941 / 940, 661 x 11008 x 1024 127.7 / 117.9, 512 x 3072 x 768 25.1 / 23.0, 8134 x 451 x
// 5225 326 / 298, 283256 x 72 x 331 197 / 137 (64 x 80 tiles; 168 with the waves 2 x 2), 361104 x 36 x 196 92 / 74 (64 x 48; 92),
// 3325 x 1824 x 328 37.8 / 35.2, 196 x 512 x 256 5.3 / 4.8, 369 x 320 x 608 8.8 / 8.3.  Behind where tiles are few and K is long (29 x 1000 x
// 11976 18.8 / 147): K groups and partitions stay sgemm.hip's.
//
// Compile-time parameters (-D, one shared library per combination):
//   BLOCK_ROWS x BLOCK_COLS   workgroup tile, of WAVES_M x 4 / WAVES_M waves, whole 16 x 16 tiles each
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <utility>

#include "helix_abi.h"
#include "helix_fastdiv.h"
#include "helix_ring.h"
#include "helix_sums.h"

#ifndef BLOCK_ROWS
#define BLOCK_ROWS 64
#endif
#ifndef BLOCK_COLS
#define BLOCK_COLS 64
#endif
#ifndef WAVES_M
#define WAVES_M 2
#endif

namespace {

using namespace helix_ring;
using helix_sums::Sums;

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int BM = BLOCK_ROWS, BN = BLOCK_COLS, WM = WAVES_M, WN = 4 / WM, TM = BM / WM / 16, TN = BN / WN / 16, NM = TM * TN, STAGES = 2, BK = 32;
constexpr int NTHREADS = 256, STEPS = BK / 8;       // k steps of four in half a K tile
constexpr int A_BYTES = BM * BK * 4, STAGE_BYTES = (BM + BN) * BK * 4, RING_BYTES = STAGES * STAGE_BYTES;
// 1 KiB copies of a K tile, dealt out to the waves, A's from wave 0 on, B's from wave 2 on.  Where a count is no multiple of four
// the waves it leaves out copy zeros to a place behind the ring: a branch among the products costs more
constexpr int PIECES_A = BM / 8, PIECES_B = BN / 8, CA = (PIECES_A + 3) / 4, CB = (PIECES_B + 3) / 4, COPIES = CA + CB;
constexpr bool EVEN = PIECES_A % 4 == 0 && PIECES_B % 4 == 0;
constexpr int LDS_BYTES = RING_BYTES + (EVEN ? 0 : 1024);
__device__ __forceinline__ int piece_of(int d, int wave) { return d < CA ? d * 4 + wave : (d - CA) * 4 + (wave ^ 2); }
__device__ __forceinline__ bool has_piece(int d, int wave) { return EVEN || piece_of(d, wave) < (d < CA ? PIECES_A : PIECES_B); }
// LDS offset of a wave's piece
__device__ __forceinline__ int place_of(int d, int wave, int stage) {
    return has_piece(d, wave) ? stage * STAGE_BYTES + (d < CA ? 0 : A_BYTES) + piece_of(d, wave) * 1024 : RING_BYTES;
}

static_assert((WM == 1 || WM == 2 || WM == 4) && BM % (16 * WM) == 0 && BN % (16 * WN) == 0, "whole 16 x 16 tiles in every wave");
static_assert(TM >= 1 && TN >= 1 && TM <= 8 && TN <= 8, "wave tiles of 16 x 16 .. 128 x 128");
static_assert(STAGES == 2 && COPIES <= 63, "the wait in a tile's middle is for every copy; a 6-bit counter");
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

// Bytes of the rows that a K tile has of an operand, from column `first` on, with `rows` of K left: an operand may have 4 GiB, a tile's
// buffer stays below the offset that reads zeros
__host__ __device__ __forceinline__ unsigned tile_bytes(int rows, int ld, int first) {
    return (unsigned)(((size_t)(rows < BK ? rows : BK) * ld - first) * 4);
}

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
template <int SUMS, int T_BM = BM, int T_BN = BN>
__global__ __launch_bounds__(NTHREADS, SUMS == helix_sums::BLOCKS ? 1 : 2) void helix_sgemm_f32_ring_kernel(const Params p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave / WN, wave_n = wave % WN, r = lane & 15, q = lane >> 4;
    int tm, tn;
    if (!tile_of((int)blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn)) return;
    const int m0 = tm * BM, n0 = tn * BN;

    // ---- copies: a stage holds 32 rows of A's BM columns, then of B's BN; a wave's piece is 64 chunks of 16 bytes of them -----
    // (whole rows of lda and ldb are inside the buffers, rows from K on are not; columns beyond M and N that lie in a chunk of the
    // last ones go into results that are not stored)
    int from[COPIES];
#pragma unroll
    for (int d = 0; d < COPIES; d++) {
        const int T = d < CA ? BM : BN, chunk = piece_of(d, wave) * 64 + lane;
        const int row = chunk / (T / 4), col = chunk % (T / 4) * 4;
        from[d] = has_piece(d, wave) && (d < CA ? m0 : n0) + col < (d < CA ? p.M : p.N) ? (row * (d < CA ? p.lda : p.ldb) + col) * 4 : OOB_OFFSET;
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)smem;
    const int ktiles = (p.K + BK - 1) / BK;
    // (past the last tile the copies still go out, from empty buffers: the counts stay)
    auto rsrc_of = [&](const float* base, int ld, int first, int t) -> intx4 {
        const int k0 = t < ktiles ? t * BK : 0;
        return raw_rsrc(base + (size_t)k0 * ld + first, t < ktiles ? tile_bytes(p.K - k0, ld, first) : 0u);
    };
    auto copy = [&](int d, int stage, const intx4& ra, const intx4& rb) {
        copy16(d < CA ? ra : rb, lds0 + (unsigned)place_of(d, wave, stage), from[d]);
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
    Sums<TM, TN, SUMS> sums;
    sums.start();
    constexpr int BLOCK = sums.BLOCK_TILES;
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
        sums.multiply(i, j, h * STEPS + s, fa[h][s][i], fb[h][s][j]);
    };
    // fragment reads that are out after g products: they end two thirds into a half
    auto due = [](int g, int reads) constexpr -> int { return 3 * g >= 2 * PRODUCTS ? reads : 3 * g * reads / (2 * PRODUCTS); };

    wait<COPIES, false>();                  // the first stage is there
    __syncthreads();
    each<READS>([&](auto e) __attribute__((always_inline)) { read(e, 0, 0); });
    int stage = 0;
    // (whole tiles, and half a one behind the loop where no more is left: a way out in the middle of the loop had the compiler copy
    // every accumulator twice a tile)
    const int halves = (p.K + BK / 2 - 1) / (BK / 2);
    for (int t = 0, end; t < halves / 2; t = end) {
        end = BLOCK && t + BLOCK < halves / 2 ? t + BLOCK : halves / 2;
        for (int u = t; u < end; u++) {
            const int next = stage + 1 == STAGES ? 0 : stage + 1;
            const intx4 ra = rsrc_of(p.A, p.lda, m0, u + STAGES), rb = rsrc_of(p.B, p.ldb, n0, u + STAGES);
            each<PRODUCTS>([&](auto g) __attribute__((always_inline)) {
                multiply(g, 0);
#pragma unroll
                for (int e = due(g, READS); e < due(g + 1, READS); e++) read(e, 1, stage);
                __builtin_amdgcn_sched_barrier(0);
            });
            // this wave is done reading tile t, and its copies of tile t + 1 have landed; behind the barrier that holds for all
            wait_and_meet<0>();
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
        if constexpr (BLOCK > 0)
            if (end < halves / 2 || ((halves & 1) && end - t == BLOCK)) sums.end_block();
    }
    if (halves & 1) each<PRODUCTS>([&](auto g) __attribute__((always_inline)) { multiply(g, 0); });
    sums.finish(halves & 1);
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
                    __builtin_nontemporal_store(floatx4{sums.sum[i][j][v], sums.sum[i][j + w / 4][v], sums.sum[i][j + w / 2][v], sums.sum[i][j + w - 1][v]},
                                                (floatx4*)dst);
                } else if (w >= 2 && vec >= 2 && col + w <= p.N) {
#pragma unroll
                    for (int e = 0; e < w; e += 2)
                        __builtin_nontemporal_store(floatx2{sums.sum[i][j + e][v], sums.sum[i][j + e + 1][v]}, (floatx2*)(dst + e));
                } else {
#pragma unroll
                    for (int e = 0; e < w; e++)
                        if (col + e < p.N) dst[e] = sums.sum[i][j + e][v];
                }
            }
        }
    }
}

// ---- convolutions --------------------------------------------------------------------------------------------------------
// The implicit GEMM: rows are pixels, columns filters, K the taps' channels, which are contiguous in both operands and stay so in
// LDS: 32 k of a row in 128 bytes, its 16-byte chunk c at c ^ (row / 2 mod 8), so that a lane reads four k of a row at once, which
// are the operands of four products.  A copy's lane knows where the first tap of its pixel lies and which taps are inside the
// image (a bit each); a tile adds the tap's offset, one for all lanes where channels come in 32s, five instructions a copy.
// Measured, us per launch, the fastest configuration of sgemm.hip and conv_patch.hip / of this (batch x channels x image, filter):
//   1x1  3 x 256 x 63 x 63 -> 96 12.6 / 10.1   3 x 128 x 49 x 49 -> 192 9.2 / 7.3     2 x 96 x 75 x 75 -> 384 15.0 / 12.5
//        41 x 128 x 45 x 45 -> 128 32.1 / 28.5  51 x 832 x 15 x 15 -> 160 37.6 / 33.8  45 x 128 x 56 x 56 -> 48 30.3 / 22.7
//   3x3  11 x 192 x 37 x 37 -> 208 107.5 / 96.2     32 x 256 x 14 x 14 -> 256 81.1 / 73.4    12 x 256 x 27 x 27 -> 160 68.6 / 63.1
//        7 x 96 x 85 x 85 -> 48 55.2 / 46.0          16 x 128 x 49 x 49 -> 64 56.1 / 51.1
//   5x5  8 x 16 x 60 x 60 -> 160 42.3 / 40.2        31 x 16 x 109 x 109 -> 48 163 / 129
// Behind, as in products, where tiles are few and K is long (1 x 256 x 14 x 14 3x3 8.0 / 20.9).

using helix_fastdiv::FastDiv;

struct ConvParams {
    const float* x;    // NHWC
    const float* w;    // [OC][kH][kW][IC]
    float* y;          // M x N
    int M, N, K, tiles_m, tiles_n;
    int H, W, IC, kH, kW, stride, pad;
    unsigned x_bytes;
    FastDiv by_OW, by_OH, by_IC, by_kW;
};
constexpr int NO_TAP = 31;                          // a bit that no row's mask has

// WHOLE: channels are a multiple of 32, so that a K tile lies in one tap
template <bool WHOLE, int SUMS, int T_BM = BM, int T_BN = BN>
__global__ __launch_bounds__(NTHREADS, SUMS == helix_sums::BLOCKS ? 1 : 2) void helix_conv_f32_ring_kernel(const ConvParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave / WN, wave_n = wave % WN, r = lane & 15, q = lane >> 4;
    int tm, tn;
    if (!tile_of((int)blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn)) return;
    const int m0 = tm * BM, n0 = tn * BN;

    // ---- copies: piece d of a wave is 8 LDS rows.  Of a pixel: where its first tap lies, and which taps are inside the image ----
    const int rows_b = (p.N - n0) < BN ? (p.N - n0) : BN;
    // (a wave's pieces are all even or all odd, so that a lane has one chunk of every row)
    const int chunk = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7);
    int first[CA];
    unsigned inside[CA];
#pragma unroll
    for (int d = 0; d < CA; d++) {
        const int m = m0 + piece_of(d, wave) * 8 + (lane >> 3);
        const int t = p.by_OW.div(m), ow = m - t * p.by_OW.d, b = p.by_OH.div(t), oh = t - b * p.by_OH.d;
        const int ih = oh * p.stride - p.pad, iw = ow * p.stride - p.pad;
        first[d] = (int)((((unsigned)b * p.H + ih) * p.W + iw) * (unsigned)p.IC * 4u) + (WHOLE ? chunk * 16 : 0);
        const int left = iw < 0 ? -iw : 0, right = p.W - iw < p.kW ? p.W - iw : p.kW;
        const unsigned of_row = right > left ? (1u << right) - (1u << left) : 0u;
        unsigned mask = 0;
        for (int kh = 0; kh < p.kH; kh++) mask |= (unsigned)(ih + kh) < (unsigned)p.H ? of_row << (kh * p.kW) : 0u;
        inside[d] = has_piece(d, wave) && m < p.M ? mask : 0u;
    }
    int of_b[CB];
#pragma unroll
    for (int d = 0; d < CB; d++) {
        const int row = piece_of(CA + d, wave) * 8 + (lane >> 3);
        of_b[d] = has_piece(CA + d, wave) && row < rows_b ? row * p.K * 4 + chunk * 16 : OOB_OFFSET;
    }
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)smem;
    const int ktiles = (p.K + BK - 1) / BK;
    const float* base_b = p.w + (size_t)n0 * p.K;
    const unsigned bytes_b = (unsigned)rows_b * (unsigned)p.K * 4u;
    const intx4 rx = raw_rsrc(p.x, p.x_bytes);
    // tap and byte offset behind a row's first tap, of the tile that is copied next: one for all lanes, or by the lane's chunk
    int tap = 0, offset = 0, kw = 0, c = 0;
    intx4 rw;
    auto aim = [&](int t) {
        rw = raw_rsrc(base_b + (size_t)(t < ktiles ? t : 0) * BK, t < ktiles ? bytes_b - (unsigned)t * (BK * 4u) : 0u);
        if (WHOLE) return;
        const int k = t * BK + chunk * 4, at = p.by_IC.div(k), row = p.by_kW.div(at);
        tap = k < p.K ? at : NO_TAP;
        offset = ((row * p.W + at - row * p.kW) * p.IC + k - at * p.IC) * 4;
    };
    auto step = [&]() {                              // WHOLE: to the next tile
        // by selection where around a branch the compiler holds the accumulators twice; elsewhere the branch is the shorter way
        if constexpr (SUMS == helix_sums::FINE || (SUMS == helix_sums::HALVES && NM > 4)) {
            const bool next_tap = c + BK == p.IC, next_row = next_tap && kw + 1 == p.kW;
            c = next_tap ? 0 : c + BK;
            tap += next_tap && tap < NO_TAP ? 1 : 0;
            kw = next_row ? 0 : next_tap ? kw + 1 : kw;
            offset += BK * 4 + (next_row ? (p.W - p.kW) * p.IC * 4 : 0);
        } else {
            c += BK;
            offset += BK * 4;
            if (c == p.IC) {
                c = 0;
                tap = tap < NO_TAP ? tap + 1 : NO_TAP;
                if (++kw == p.kW) {
                    kw = 0;
                    offset += (p.W - p.kW) * p.IC * 4;
                }
            }
        }
    };
    auto copy = [&](int d, int stage) {
        const unsigned to = lds0 + (unsigned)place_of(d, wave, stage);
        if (d < CA) copy16(rx, to, (inside[d] >> tap) & 1 ? first[d] + offset : OOB_OFFSET);
        else copy16(rw, to, !WHOLE && tap == NO_TAP ? OOB_OFFSET : of_b[d - CA]);
    };
#pragma unroll
    for (int u = 0; u < STAGES; u++) {
        aim(u);
#pragma unroll
        for (int d = 0; d < COPIES; d++) copy(d, u);
        if (WHOLE) step();
    }

    // ---- fragments: lane (r, q) supplies row r, chunk 4 h + q of half h ------------------------------------------------
    int at_a[2], at_b[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int chunk = ((h * 4 + q) ^ (r >> 1)) << 4;
        at_a[h] = (wave_m * TM * 16 + r) * BK * 4 + chunk;
        at_b[h] = A_BYTES + (wave_n * TN * 16 + r) * BK * 4 + chunk;
    }
    Sums<TM, TN, SUMS> sums;
    sums.start();
    constexpr int BLOCK = sums.BLOCK_TILES;
    floatx4 fa[2][TM], fb[2][TN];
    constexpr int READS = TM + TN, PRODUCTS = 4 * NM;
    auto read = [&](int e, int h, int stage) {
        const unsigned char* from = smem + stage * STAGE_BYTES;
        if (e < TM) fa[h][e] = *(const floatx4*)(from + at_a[h] + e * 16 * BK * 4);
        else fb[h][e - TM] = *(const floatx4*)(from + at_b[h] + (e - TM) * 16 * BK * 4);
    };
    // the filters go first, which leaves a lane with four consecutive columns of one row
    auto multiply = [&](int g, int h) {
        const int e = g / NM, i = g % NM % TM, j = g % NM / TM;
        sums.multiply(i, j, h * 4 + e, fb[h][j][e], fa[h][i][e]);
    };
    auto due = [](int g, int reads) constexpr -> int { return 3 * g >= 2 * PRODUCTS ? reads : 3 * g * reads / (2 * PRODUCTS); };

    wait<COPIES, false>();                  // the first stage is there
    __syncthreads();
    each<READS>([&](auto e) __attribute__((always_inline)) { read(e, 0, 0); });
    int stage = 0;
    const int halves = (p.K + BK / 2 - 1) / (BK / 2);       // as in the products' loop
    for (int t = 0, end; t < halves / 2; t = end) {
        end = BLOCK && t + BLOCK < halves / 2 ? t + BLOCK : halves / 2;
        for (int u = t; u < end; u++) {
            const int next = stage + 1 == STAGES ? 0 : stage + 1;
            each<PRODUCTS>([&](auto g) __attribute__((always_inline)) {
                multiply(g, 0);
#pragma unroll
                for (int e = due(g, READS); e < due(g + 1, READS); e++) read(e, 1, stage);
                __builtin_amdgcn_sched_barrier(0);
            });
            aim(u + STAGES);
            wait_and_meet<0>();
            each<PRODUCTS>([&](auto g) __attribute__((always_inline)) {
                multiply(g, 1);
#pragma unroll
                for (int e = due(g, READS); e < due(g + 1, READS); e++) read(e, 0, next);   // (past the last tile: zeros, not used)
#pragma unroll
                for (int d = g * COPIES / PRODUCTS; d < (g + 1) * COPIES / PRODUCTS; d++) copy(d, stage);
                __builtin_amdgcn_sched_barrier(0);
            });
            if (WHOLE) step();
            stage = next;
        }
        if constexpr (BLOCK > 0)
            if (end < halves / 2 || ((halves & 1) && end - t == BLOCK)) sums.end_block();
    }
    if (halves & 1) each<PRODUCTS>([&](auto g) __attribute__((always_inline)) { multiply(g, 0); });
    sums.finish(halves & 1);
    wait<0, true>();                                 // no copy is left when the workgroup gives its LDS back

    // ---- results: a quarter's lanes hold 16 bytes of 16 rows ---------------------------------------------------------------
    const bool wide = (((uintptr_t)p.y >> 2 | (unsigned)p.N) & 3) == 0;
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int row = m0 + (wave_m * TM + i) * 16 + r;
        if (row >= p.M) continue;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col = n0 + (wave_n * TN + j) * 16 + 4 * q;
            float* dst = p.y + (size_t)row * p.N + col;
            if (wide && col + 4 <= p.N) {
                __builtin_nontemporal_store(sums.sum[i][j], (floatx4*)dst);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (col + e < p.N) dst[e] = sums.sum[i][j][e];
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
                 "\"k_multiple\": 1, \"ld_multiple\": 4, \"conv\": \"NHWC x [OC][kH][kW][IC]; IC a multiple of 4, at most 31 taps\"}",
                 STAGES, BM, BN, BM / WM, BN / WN, BK, NTHREADS, LDS_BYTES);
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

template <int SUMS>
inline int launch_gemm(const Params& p, unsigned grid, hipStream_t s) {
    static int rc = (int)hipFuncSetAttribute((const void*)helix_sgemm_f32_ring_kernel<SUMS>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
    if (rc) return rc;
    hipLaunchKernelGGL(helix_sgemm_f32_ring_kernel<SUMS>, dim3(grid), dim3(NTHREADS), LDS_BYTES, s, p);
    return (int)hipGetLastError();
}

// Rows of `ld` floats as an operand: byte offsets inside one K tile are 31-bit, in all as sgemm.hip takes them
inline bool operand_fits(int K, int ld) { return (long long)K * ld * 4 < 0xffffffffLL && (long long)BK * ld * 4 < 0x7fffffffLL; }

inline int gemm(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc, void*, size_t, hipStream_t s) {
    if (lda % 4 != 0 || ldb % 4 != 0) return HELIX_ERR_INVALID_VALUE;  // 16-byte copies along M and N
    if (lda < M || ldb < N || ldc < N) return HELIX_ERR_INVALID_VALUE;
    if (((uintptr_t)A & 15) || ((uintptr_t)B & 15) || ((uintptr_t)C & 3)) return HELIX_ERR_INVALID_VALUE;
    if (!operand_fits(K, lda) || !operand_fits(K, ldb)) return HELIX_ERR_INVALID_VALUE;
    Params p{(const float*)A, (const float*)B, (float*)C, M, N, K, lda, ldb, ldc, (M - 1) / BM + 1, (N - 1) / BN + 1};
    const long long ntiles = (long long)p.tiles_m * p.tiles_n;
    if (ntiles > 0x3fffffffLL) return HELIX_ERR_INVALID_VALUE;
    const unsigned grid = (unsigned)((ntiles + NUM_XCD - 1) / NUM_XCD * NUM_XCD);
    switch (helix_sums::mode_of(M, N, K)) {
        case helix_sums::FINE: return launch_gemm<helix_sums::finest(TM, TN)>(p, grid, s);
        case helix_sums::HALVES: return launch_gemm<helix_sums::HALVES>(p, grid, s);
        default: return launch_gemm<helix_sums::BLOCKS>(p, grid, s);
    }
}

template <bool WHOLE, int SUMS>
inline int launch_conv(const ConvParams& p, unsigned grid, hipStream_t s) {
    static int rc = (int)hipFuncSetAttribute((const void*)helix_conv_f32_ring_kernel<WHOLE, SUMS>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
    if (rc) return rc;
    hipLaunchKernelGGL((helix_conv_f32_ring_kernel<WHOLE, SUMS>), dim3(grid), dim3(NTHREADS), LDS_BYTES, s, p);
    return (int)hipGetLastError();
}

template <int SUMS>
inline int launch_conv(const ConvParams& p, unsigned grid, hipStream_t s) {
    return p.IC % BK == 0 ? launch_conv<true, SUMS>(p, grid, s) : launch_conv<false, SUMS>(p, grid, s);
}

inline int conv2d(const void* x, const void* w, void* y, int batch, int H, int W, int IC, int OC, int kH, int kW, int stride,
                  int pad, void*, size_t, hipStream_t s) {
    if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)y & 3)) return HELIX_ERR_INVALID_VALUE;
    const int OH = (H + 2 * pad - kH) / stride + 1, OW = (W + 2 * pad - kW) / stride + 1;
    // a 16-byte chunk lies in one tap, and a row's mask has a bit for each and one to spare
    if (IC % 4 != 0 || kH > NO_TAP || kW > NO_TAP || kH * kW > NO_TAP) return HELIX_ERR_UNSUPPORTED;
    const long long M = (long long)batch * OH * OW, K = (long long)kH * kW * IC;
    const long long xbytes = (long long)batch * H * W * IC * 4;
    if (M > 0x7fffffffLL - BM || K > 0x7fffffffLL - 4 * BK || xbytes >= 0x7fffffffLL) return HELIX_ERR_INVALID_VALUE;
    if ((long long)BN * K * 4 >= 0x7fffffffLL) return HELIX_ERR_INVALID_VALUE;
    ConvParams p{(const float*)x, (const float*)w, (float*)y, (int)M, OC, (int)K, ((int)M - 1) / BM + 1, (OC - 1) / BN + 1,
                 H, W, IC, kH, kW, stride, pad, (unsigned)xbytes,
                 helix_fastdiv::make(OW), helix_fastdiv::make(OH), helix_fastdiv::make(IC), helix_fastdiv::make(kW)};
    const long long ntiles = (long long)p.tiles_m * p.tiles_n;
    if (ntiles > 0x3fffffffLL) return HELIX_ERR_INVALID_VALUE;
    const unsigned grid = (unsigned)((ntiles + NUM_XCD - 1) / NUM_XCD * NUM_XCD);
    switch (helix_sums::mode_of(M, OC, K)) {
        case helix_sums::FINE: return launch_conv<helix_sums::finest(TM, TN)>(p, grid, s);
        case helix_sums::HALVES: return launch_conv<helix_sums::HALVES>(p, grid, s);
        default: return launch_conv<helix_sums::BLOCKS>(p, grid, s);
    }
}

}  // namespace tpl

#define HELIX_TPL_SCRATCH_BYTES 256   // this family never asks for a workspace
#include "helix_host.h"
