// The FP32 sums of one wave's tiles of v_mfma_f32_16x16x4_f32 products (MI355X_FP32/gemm_ring.hip, common/helix_conv_patch.h).
//
// A sum of K products leaves an error that grows with the root of the products in a chain and of the partial sums that are added in
// turn: about 0.18e-7 x sqrt(chain + partial sums) in the norm, against 64 bits, operands ~ N(0, 1).  The K groups and K partitions of
// sgemm.hip and the lanes of the GEMV keep both short on small problems; what takes their place has to, too.
// Error x 1e7 of the fastest configuration of those / one chain / these:
//   BLOCKS  a chain per 256 of K, in order                     4000 x 2300 x 770 4.8 / 5.0 / 2.9; 422 x 4016 x 4456 8.5 / 12 / 3.0
//   HALVES  a chain per 16                                     196 x 512 x 256 1.5 / 2.9 / 1.1; 314 x 360 x 776 1.6 / 5.0 / 1.5
//   FINE    chains of 8, added over 32, those with what each addition loses added up beside    40000 x 7 x 500 0.85 / 4.0 / 0.73
//   TILES   a chain per 32, where there are no registers for HALVES
// HALVES takes 2 - 4 % of the time of a launch that BLOCKS would do (196 x 512 x 256 4.7 / 4.8 us, 369 x 320 x 608 7.8 / 8.1; wave tiles of
// six and more 5 %), FINE 5 % on the tall products that it is for (14.2 / 15.0).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace helix_sums {

typedef float floatx4 __attribute__((ext_vector_type(4)));

enum { CHAIN, BLOCKS, TILES, HALVES, FINE };         // CHAIN: one for all of K (products of 16-bit operands)

template <int TM, int TN>
using Tiles = floatx4[TM][TN];

template <int TM, int TN>
__device__ __forceinline__ void clear(Tiles<TM, TN>& acc) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
}

template <int TM, int TN>
__device__ __forceinline__ void add(Tiles<TM, TN>& sum, const Tiles<TM, TN>& acc) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) sum[i][j] += acc[i][j];
}

// (products of 16-bit operands, which the caller writes himself)
template <int TM, int TN>
struct ChainSums {
    static constexpr int BLOCK_TILES = 0;
    Tiles<TM, TN> sum;
    __device__ __forceinline__ void start() { clear<TM, TN>(sum); }
    __device__ __forceinline__ void finish(bool) {}
};

template <int TM, int TN, int TILES_>
struct BlockSums {
    static constexpr int BLOCK_TILES = TILES_;
    Tiles<TM, TN> acc, sum;                          // of this block of K, of the blocks before it
    __device__ __forceinline__ void start() {
        clear<TM, TN>(acc);
        clear<TM, TN>(sum);
    }
    // product `step` (0 .. 7) of a K tile
    __device__ __forceinline__ void multiply(int i, int j, int, float b, float a) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b, a, acc[i][j], 0, 0, 0);
    }
    __device__ __forceinline__ void end_block() {
        add<TM, TN>(sum, acc);
        clear<TM, TN>(acc);
    }
    __device__ __forceinline__ void finish(bool) { add<TM, TN>(sum, acc); }
};

template <int TM, int TN>
struct HalfSums {
    static constexpr int BLOCK_TILES = 0;             // no blocks
    // of a half, of the halves before it.  A wave of one tile has two in turn and adds one a product into the other: it would wait for
    // the product before it otherwise, where others have a round of products in between
    static constexpr int TURNS = TM * TN == 1 ? 2 : 1;
    Tiles<TM, TN> acc[TURNS], sum;
    __device__ __forceinline__ void start() {
#pragma unroll
        for (int t = 0; t < TURNS; t++) clear<TM, TN>(acc[t]);
        clear<TM, TN>(sum);
    }
    __device__ __forceinline__ void multiply(int i, int j, int step, float b, float a) {
        floatx4& to = acc[step / 4 % TURNS][i][j];
        if (step % 4 == 0) {
            if (TURNS == 1) sum[i][j] += to;
            to = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        to = __builtin_amdgcn_mfma_f32_16x16x4f32(b, a, to, 0, 0, 0);
        if (TURNS == 2 && step % 4 == 1) sum[i][j] += acc[(step / 4 + 1) % TURNS][i][j];
    }
    __device__ __forceinline__ void finish(bool half) {     // half: the last tile had its first half only
        if (TURNS == 1 || half) add<TM, TN>(sum, acc[0]);
        else add<TM, TN>(sum, acc[TURNS - 1]);
    }
};

template <int TM, int TN>
struct FineSums {
    static constexpr int BLOCK_TILES = 0;             // no blocks
    Tiles<TM, TN> acc, tile, sum, low;               // of a chain that is not a tile's first, of a tile, of the tiles before it; what sum lost
    __device__ __forceinline__ void start() {
        clear<TM, TN>(acc);
        clear<TM, TN>(tile);
        clear<TM, TN>(sum);
        clear<TM, TN>(low);
    }
    // What an addition loses is added up beside the sum, the Kahan-Babuska way, and not taken off the next tile as Kahan does: there an infinite
    // sum would be NaN behind the next one (inf - inf), and asking for that each time costs 1 - 8 %
    __device__ __forceinline__ void add_tile(int i, int j) {
        const floatx4 t = sum[i][j] + tile[i][j];
        low[i][j] += tile[i][j] - (t - sum[i][j]);
        sum[i][j] = t;
    }
    // a chain is added when the next one begins, a round of products later
    __device__ __forceinline__ void multiply(int i, int j, int step, float b, float a) {
        floatx4& to = step < 2 ? tile[i][j] : acc[i][j];
        if (step % 2 == 0) {
            if (step != 2) tile[i][j] += acc[i][j];
            if (step == 0) add_tile(i, j);
            to = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        to = __builtin_amdgcn_mfma_f32_16x16x4f32(b, a, to, 0, 0, 0);
    }
    __device__ __forceinline__ void finish(bool) {
        add<TM, TN>(tile, acc);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                add_tile(i, j);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (__builtin_fabsf(sum[i][j][e]) < __builtin_inff()) sum[i][j][e] += low[i][j][e];
            }
    }
};

// FINE's four sets of accumulators are for wave tiles of up to four, which the few rows or columns that it is for are run on.  FINE and HALVES
// are for kernels of at most 256 registers: beyond them the compiler keeps accumulators where VALU instructions do not read them.
constexpr int finest(int tm, int tn) { return tm * tn <= 4 ? FINE : HALVES; }
template <int TM, int TN, int MODE>
using Sums = std::conditional_t<MODE == CHAIN, ChainSums<TM, TN>, std::conditional_t<MODE == BLOCKS || MODE == TILES, BlockSums<TM, TN, MODE == BLOCKS ? 8 : 1>,
             std::conditional_t<MODE == HALVES, HalfSums<TM, TN>, FineSums<TM, TN>>>>;

// How an M x N result of K products each is summed, K in `parts` that have sums of their own.  K groups of four and more, or partitions, were
// the fastest of sgemm.hip up to 2^20 results, two groups up to 4.6e6 (their chains are no shorter than BLOCKS' from K = 512 on), GEMVs
// up to 16 rows or columns, of 130 problems; beyond K = 2048 HALVES adds as many partial sums as BLOCKS has products in a chain.
inline int mode_of(long long M, long long N, long long K, int parts = 1) {
    const long long results = M * N;
    if ((M <= 16 || N <= 16) && K >= 256) return FINE;
    return K / parts <= 2048 && (results <= 1LL << 20 || (results <= 5LL << 20 && K < 512)) ? HALVES : BLOCKS;
}

}  // namespace helix_sums
