// MI355X (gfx950 / CDNA4) FP16 convolution template whose input stays in LDS while the filter walks over it.
//
//   y[B,OH,OW,OC] = conv2d(x[B,H,W,IC], w[OC,kH,kW,IC]), IC a multiple of 8.  FP16 in, FP32 accumulate (MFMA), FP16 out.
//
// Role in the reference: the im2col.cu + gemm.cu pair (src_template/Ampere_FP16/im2col.cu:38-97), as the implicit GEMM of
// gemm.hip; this family is for the layers that one is slow on.
//
// What bounds those: gemm.hip gathers a tile's rows from L2 again for every filter tap, and a compute unit takes 46 bytes per
// clock from there, so that a 64 x 64 tile is fed in 2.8 times the time it multiplies; and a layer of few output tiles and
// long K has to be cut along K over workgroups, whose sums meet in a tail of 3.3 us.  Here
//   * a workgroup stages the input rows under its BLOCK_ROWS output pixels in LDS once, with all channels and with the
//     padding, and every tap of the filter reads them there: 16 pixels x 32 channels of one tap are the MFMA's operand, at
//     an LDS offset from each pixel's corner that a table holds (K in chunks of eight channels, any number of them);
//   * K_GROUPS waves share each output tile, each with its part of K, and add their sums through LDS, in order: the few
//     workgroups of a small layer keep their compute units busy, without a second pass over memory;
//   * a wave loads its weights by itself, AHEAD K tiles in front of their use, in rows of 128 bytes, and brings them into the
//     MFMA's order through a piece of LDS that is its own: no barrier between the first product and the last.  (Loaded in the
//     MFMA's order, 16 rows x 64 bytes per instruction, they come at a quarter of the rate: 15.7 instead of 53 bytes per clock
//     and CU, one cache line looked up for each lane.)
//   * results leave from registers, 16 bytes per lane.
//
// Measured (us per launch, the fastest configuration of gemm.hip / of this family; the layer's batch, channels, image, filter):
//   4 x 256 x 14 x 14 3x3 -> 256 10.1 / 6.6     2 x 512 x 16 x 16 3x3 -> 256 10.1 / 7.4     2 x 112 x 14 x 14 3x3 -> 208 7.4 / 5.1
//   1 x 256 x 13 x 13 3x3 -> 160 7.7 / 5.6      2 x 96 x 15 x 15 5x5 -> 512 9.4 / 7.1       4 x 192 x 9 x 9 3x3 -> 48 6.7 / 5.0
//   32 x 64 x 56 x 56 3x3 -> 64 15.1 / 14.3     32 x 256 x 14 x 14 3x3 -> 256 15.2 / 13.7   16 x 48 x 40 x 40 5x5 -> 96 13.0 / 11.4
// Slower: filters with stride 2 on large images, and images or channel counts that leave room for few pixels in LDS (9 x 96 x
// 106 x 106 3x3 -> 128 32 / 50); the selection times both.  Strips of columns and passes over the channels, which would fit
// those, were built and measured: never ahead of gemm.hip there, and half a microsecond slower everywhere else.
//
// Compile-time parameters (-D, one shared library per combination):
//   BLOCK_ROWS x BLOCK_COLS   output pixels x channels of a workgroup
//   WAVE_ROWS  x WAVE_COLS    of a wave, multiples of 16
//   K_GROUPS                  parts of K, each on its own wave
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "helix_abi.h"
#include "helix_fastdiv.h"

#ifndef BLOCK_ROWS
#define BLOCK_ROWS 32
#endif
#ifndef BLOCK_COLS
#define BLOCK_COLS 32
#endif
#ifndef WAVE_ROWS
#define WAVE_ROWS 32
#endif
#ifndef WAVE_COLS
#define WAVE_COLS 32
#endif
#ifndef K_GROUPS
#define K_GROUPS 8
#endif

namespace {

using helix_fastdiv::FastDiv;
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

constexpr int TM = WAVE_ROWS / 16, TN = WAVE_COLS / 16;          // MFMA tiles of a wave
constexpr int WAVES_M = BLOCK_ROWS / WAVE_ROWS, WAVES_N = BLOCK_COLS / WAVE_COLS;
constexpr int NWAVES = WAVES_M * WAVES_N * K_GROUPS, NTHREADS = 64 * NWAVES;
constexpr int KT = 64, KT_CHUNKS = KT / 8;    // K tile: what a wave loads of its weights at a time, two MFMA steps
constexpr int AHEAD = 2;                      // K tiles of weights in flight in registers
constexpr int OWN_BYTES = WAVE_COLS * KT * 2; // a wave's piece of LDS for its weights
constexpr int SUM_BYTES = K_GROUPS > 1 ? NWAVES * TM * TN * 1024 : 0;
constexpr int LDS_MAX = 160 * 1024;
constexpr int NUM_XCD = 8;
constexpr int OOB = 0x40000000;               // byte offset beyond any buffer (they stay below it), twice too: the load returns zeros

static_assert(BLOCK_ROWS % WAVE_ROWS == 0 && BLOCK_COLS % WAVE_COLS == 0 && WAVE_ROWS % 16 == 0 && WAVE_COLS % 16 == 0, "tiles");
static_assert(TN == 1 || TN % 2 == 0, "a lane's results are four channels of a single tile or eight of a pair");
static_assert(NTHREADS <= 512 && SUM_BYTES <= LDS_MAX, "workgroup");

struct Params {
    const _Float16* x;   // NHWC
    const _Float16* w;   // [OC][kH][kW][IC]
    _Float16* y;         // NHWC
    int H, W, OH, OC, stride, pad, kW;
    int M;                                 // output pixels of the batch
    int group;                             // 16-byte chunks of a pixel's channels
    int chunks, ktiles, tiles_per_part;    // K in 16-byte chunks, in 64-wide tiles, and the tiles of one wave's part
    int blocks, blocks_per_xcd, channel_blocks;
    int image_rows;                        // staged rows of an image: (OH - 1) * stride + kH
    int row_pixels, real_pixels;           // staged pixels of a row, and those of them inside the image
    int row_chunks;                        // 16-byte chunks of the latter
    int pixel_bytes, row_bytes, patch_offset;
    int wide;                              // results leave 16 (8) bytes at a time: OC a multiple of 8 (4) and y aligned to it
    unsigned x_bytes, w_bytes;
    FastDiv by_OW, by_OH, by_group, by_kW, by_row_chunks, by_image_rows, by_channel_blocks, by_border;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ uintx4 load16(__amdgpu_buffer_rsrc_t r, int at) {
    return __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0));
}

// n / d: the bits of FastDiv::div through the high word of one 32-bit product, which the staging loop's three divisions a chunk
// are a third of.
__device__ __forceinline__ int quotient(const FastDiv& d, int n) { return (int)(__umulhi((unsigned)n << 1, d.mul) >> (d.shift - 31)); }

// Output channel (within a wave's) of row r of MFMA tile j: two tiles leave a lane of quarter q with the channels
// 8 q .. 8 q + 7 of their 32, a single one with 4 q .. 4 q + 3 of its 16.
__device__ __forceinline__ int channel_of(int j, int r) {
    return TN % 2 ? j * 16 + r : (j >> 1) * 32 + (r >> 2) * 8 + (j & 1) * 4 + (r & 3);
}

// Pixel (within an MFMA tile) of lane l.  ds_read_b128 serves lanes {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same of the
// upper half together.
__device__ __forceinline__ int pixel_of(int r) { return r < 4 ? r : r < 12 ? r + 4 : r - 8; }

// (the tile parameters are template arguments for the symbol name's sake: a profiler lists configurations separately)
template <int T_BM = BLOCK_ROWS, int T_BN = BLOCK_COLS, int T_WM = WAVE_ROWS, int T_WN = WAVE_COLS, int T_KG = K_GROUPS>
__global__ __launch_bounds__(NTHREADS, 2) void helix_conv_patch_f16_kernel(const Params p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int block = (int)(blockIdx.x % NUM_XCD) * p.blocks_per_xcd + (int)(blockIdx.x / NUM_XCD);
    if (block >= p.blocks) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int part = wave % K_GROUPS, wave_n = (wave / K_GROUPS) % WAVES_N, wave_m = wave / (K_GROUPS * WAVES_N);
    const int px_block = quotient(p.by_channel_blocks, block);
    const int oc0 = (block - px_block * p.channel_blocks) * BLOCK_COLS + wave_n * WAVE_COLS;
    const int m0 = px_block * BLOCK_ROWS;
    const int m_last = (m0 + BLOCK_ROWS < p.M ? m0 + BLOCK_ROWS : p.M) - 1;

    // ---- weights: loaded in whole 128-byte rows, AHEAD K tiles in front of their use, and brought into the MFMA's order
    // through a piece of LDS of the wave's own ---------------------------------------------------------------------------
    const int t_begin = part * p.tiles_per_part < p.ktiles ? part * p.tiles_per_part : p.ktiles;
    const int t_end = t_begin + p.tiles_per_part < p.ktiles ? t_begin + p.tiles_per_part : p.ktiles;
    const int chunk_end = KT_CHUNKS * t_end < p.chunks ? KT_CHUNKS * t_end : p.chunks;
    const __amdgpu_buffer_rsrc_t rw = rsrc(p.w, p.w_bytes);
    int w_at[2 * TN];                    // 8 rows of a tile at a time: lane l takes chunk l % 8 of row l / 8
#pragma unroll
    for (int d = 0; d < 2 * TN; d++) {
        const int n = oc0 + channel_of(d >> 1, (d & 1) * 8 + (lane >> 3));
        w_at[d] = n < p.OC ? (n * p.chunks + (lane & 7)) * 16 : OOB;
    }
    auto tile_offset = [&](int t) -> int { return KT_CHUNKS * t + (lane & 7) < chunk_end ? t * (KT * 2) : OOB; };
    uintx4 st[AHEAD][2 * TN];
#pragma unroll
    for (int u = 0; u < AHEAD; u++) {
        const int k_at = tile_offset(t_begin + u);
#pragma unroll
        for (int d = 0; d < 2 * TN; d++) st[u][d] = load16(rw, w_at[d] + k_at);
    }

    // ---- input under the block -----------------------------------------------------------------------------------------
    auto staged_row = [&](int m, int* ow) -> int {          // first staged row of an output pixel, over all images
        const int t = quotient(p.by_OW, m);
        *ow = m - __mul24(t, p.by_OW.d);
        const int image = quotient(p.by_OH, t);
        return __mul24(image, p.image_rows) + __mul24(t - __mul24(image, p.OH), p.stride);
    };
    int unused;
    const int row0 = __builtin_amdgcn_readfirstlane(staged_row(m0, &unused));
    const int kH = p.image_rows - (p.OH - 1) * p.stride;
    const int rows = __builtin_amdgcn_readfirstlane(staged_row(m_last, &unused)) + kH - row0;
    unsigned char* patch = smem + p.patch_offset;
    {
        const __amdgpu_buffer_rsrc_t rx = rsrc(p.x, p.x_bytes);
        const int total = rows * p.row_chunks, gap = p.pixel_bytes - p.group * 16, image_row_bytes = p.W * p.group * 16;
        constexpr int BATCH = 8;                            // loads of a thread in flight
        for (int i0 = tid; i0 < total; i0 += NTHREADS * BATCH) {
            uintx4 v[BATCH];
            int dst[BATCH];
#pragma unroll
            for (int u = 0; u < BATCH; u++) {
                const int i = i0 + u * NTHREADS;
                const int row = quotient(p.by_row_chunks, i), c = i - __mul24(row, p.row_chunks);
                const int image = quotient(p.by_image_rows, row0 + row), ih = row0 + row - __mul24(image, p.image_rows) - p.pad;
                const bool inside = (i < total) & ((unsigned)ih < (unsigned)p.H);
                v[u] = load16(rx, inside ? __mul24(__mul24(image, p.H) + ih, image_row_bytes) + c * 16 : OOB);
                dst[u] = i < total ? __mul24(row, p.row_bytes) + c * 16 + __mul24(quotient(p.by_group, c), gap) : -1;
            }
            unsigned char* first = patch + p.pad * p.pixel_bytes;
#pragma unroll
            for (int u = 0; u < BATCH; u++)
                if (dst[u] >= 0) *(uintx4*)(first + dst[u]) = v[u];
        }
        if (p.row_pixels > p.real_pixels) {                 // columns of padding
            const int border = p.by_border.d;               // 16-byte chunks of them per row
            for (int i = tid; i < rows * border; i += NTHREADS) {
                const int row = quotient(p.by_border, i), c = i - __mul24(row, border);
                int px = quotient(p.by_group, c);
                const int g = c - __mul24(px, p.group);
                if (px >= p.pad) px += p.real_pixels;
                *(uintx4*)(patch + row * p.row_bytes + px * p.pixel_bytes + g * 16) = uintx4{0, 0, 0, 0};
            }
        }
        // the chunk behind each pixel's channels: what K chunks beyond the filter read
        if (p.chunks % KT_CHUNKS)
            for (int i = tid; i < rows * p.row_pixels; i += NTHREADS)
                *(uintx4*)(patch + i * p.pixel_bytes + p.group * 16) = uintx4{0, 0, 0, 0};
        // LDS offset of each K chunk from a pixel's corner
        for (int j = tid; j < KT_CHUNKS * (p.ktiles + 1); j += NTHREADS) {
            const int tap = quotient(p.by_group, j), g = j - __mul24(tap, p.group);
            const int kh = quotient(p.by_kW, tap), kw = tap - __mul24(kh, p.kW);
            ((int*)(smem + NWAVES * OWN_BYTES))[j] = j < p.chunks ? __mul24(kh, p.row_bytes) + __mul24(kw, p.pixel_bytes) + g * 16
                                                              : p.chunks % KT_CHUNKS ? p.group * 16 : 0;
        }
    }
    int at[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        int m = m0 + (wave_m * TM + i) * 16 + pixel_of(r), ow;
        m = m < m_last ? m : m_last;
        const int row = staged_row(m, &ow) - row0;
        at[i] = p.patch_offset + __mul24(row, p.row_bytes) + __mul24(ow, p.stride * p.pixel_bytes);
    }
    __syncthreads();

    // ---- products ----------------------------------------------------------------------------------------------------
    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int* table = (const int*)(smem + NWAVES * OWN_BYTES) + q;
    // rows of 128 bytes, 16-byte chunk c of row r at c ^ (r / 2 mod 8): reads and writes free of bank conflicts
    unsigned char* own = smem + wave * OWN_BYTES;
    unsigned char* own_write = own + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 4)) << 4);
    unsigned char* own_write_odd = own + (lane >> 3) * 128 + (((lane & 7) ^ ((lane >> 4) + 4)) << 4);
    auto write_b = [&](int d, uintx4 v) { *(uintx4*)((d & 1 ? own_write_odd : own_write) + d * 1024) = v; };
    auto read_b = [&](int s, int j) -> half8 { return *(const half8*)(own + j * 2048 + r * 128 + (((s * 4 + q) ^ (r >> 1)) << 4)); };
    half8 a[2][TM], b[2][TN];
    int off;
    constexpr int SLOTS = TM * TN;
    // One K tile, st holding the weights of the next one.  Behind each MFMA its share of the other instructions: the reads of
    // the second step's operands behind the first step's, of the next tile's first step's behind the second step's, once its
    // weights have taken this tile's place (a wave's LDS instructions execute in their order), and the loads AHEAD tiles on.
    auto tile = [&](int t, uintx4 (&stv)[2 * TN]) {
        const int k_at = tile_offset(t + 1 + AHEAD);
#pragma unroll
        for (int g = 0; g < SLOTS; g++) {
            const int i = g % TM, j = g / TM;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[0][j], a[0][i], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int e = 0; e < TM + TN + 1; e++) {
                if (e * SLOTS / (TM + TN + 1) != g) continue;
                if (e < TM) a[1][e] = *(const half8*)(smem + at[e] + off);
                else if (e == TM) off = table[KT_CHUNKS * (t + 1)];
                else b[1][e - TM - 1] = read_b(1, e - TM - 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int g = 0; g < SLOTS; g++) {
            const int i = g % TM, j = g / TM;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[1][j], a[1][i], acc[i][j], 0, 0, 0);
            constexpr int W = 2 * TN, COUNT = 2 * W + TM + TN + 1;
#pragma unroll
            for (int e = 0; e < COUNT; e++) {
                if (e * SLOTS / COUNT != g) continue;
                if (e < W) write_b(e, stv[e]);
                else if (e < W + TM) a[0][e - W] = *(const half8*)(smem + at[e - W] + off);
                else if (e == W + TM) off = table[KT_CHUNKS * (t + 1) + 4];
                else if (e < W + TM + 1 + TN) b[0][e - W - TM - 1] = read_b(0, e - W - TM - 1);
                else stv[e - W - TM - TN - 1] = load16(rw, w_at[e - W - TM - TN - 1] + k_at);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // the first tile's operands; its registers take tile AHEAD
    {
        const int k_at = tile_offset(t_begin + AHEAD);
#pragma unroll
        for (int d = 0; d < 2 * TN; d++) {
            write_b(d, st[0][d]);
            st[0][d] = load16(rw, w_at[d] + k_at);
        }
        off = table[KT_CHUNKS * t_begin];
#pragma unroll
        for (int i = 0; i < TM; i++) a[0][i] = *(const half8*)(smem + at[i] + off);
#pragma unroll
        for (int j = 0; j < TN; j++) b[0][j] = read_b(0, j);
        off = table[KT_CHUNKS * t_begin + 4];
    }
    int t = t_begin;
    for (; t + AHEAD <= t_end; t += AHEAD) {
        tile(t, st[1]);
        tile(t + 1, st[0]);
    }
    if (t < t_end) tile(t, st[1]);

    // ---- results -----------------------------------------------------------------------------------------------------
    constexpr int PAIR = TN % 2 ? 1 : 2, UNITS = TM * (TN / PAIR);
    auto store = [&](int i, int jj, const floatx4 (&v)[PAIR]) {
        const int m = m0 + (wave_m * TM + i) * 16 + pixel_of(r);
        if (m > m_last) return;
        const int n = oc0 + jj * (16 * PAIR) + q * (4 * PAIR);
        _Float16* dst = p.y + (size_t)m * p.OC + n;
        _Float16 h[4 * PAIR];
#pragma unroll
        for (int e = 0; e < 4 * PAIR; e++) h[e] = (_Float16)v[e >> 2][e & 3];
        if (p.wide) {
            if (n < p.OC) {
                if constexpr (PAIR == 2) *(half8*)dst = half8{h[0], h[1], h[2], h[3], h[4], h[5], h[6], h[7]};
                else *(half4*)dst = half4{h[0], h[1], h[2], h[3]};
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4 * PAIR; e++)
                if (n + e < p.OC) dst[e] = h[e];
        }
    };
    if constexpr (K_GROUPS == 1) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int jj = 0; jj < TN / PAIR; jj++) {
                floatx4 v[PAIR];
#pragma unroll
                for (int e = 0; e < PAIR; e++) v[e] = acc[i][jj * PAIR + e];
                store(i, jj, v);
            }
    } else {
        // parts of K: added through LDS in their order, the units of a wave's tile shared out over its parts
        __syncthreads();
        floatx4* sums = (floatx4*)smem + (size_t)(wave_m * WAVES_N + wave_n) * K_GROUPS * (TM * TN * 64);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) sums[(part * (TM * TN) + i * TN + j) * 64 + lane] = acc[i][j];
        __syncthreads();
        for (int u = part; u < UNITS; u += K_GROUPS) {
            const int i = u / (TN / PAIR), jj = u % (TN / PAIR);
            floatx4 v[PAIR];
#pragma unroll
            for (int e = 0; e < PAIR; e++) v[e] = sums[(i * TN + jj * PAIR + e) * 64 + lane];
            for (int k = 1; k < K_GROUPS; k++)
#pragma unroll
                for (int e = 0; e < PAIR; e++) v[e] += sums[(k * (TM * TN) + i * TN + jj * PAIR + e) * 64 + lane];
            store(i, jj, v);
        }
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
                 "{\"family\": \"gemm_f16\", \"input_in_lds\": 1, \"arch\": \"gfx950\", \"mfma\": \"v_mfma_f32_16x16x32_f16\", "
                 "\"block_rows\": %d, \"block_cols\": %d, \"wave_rows\": %d, \"wave_cols\": %d, \"block_k\": %d, "
                 "\"k_groups\": %d, \"split_k\": 1, \"threads\": %d, \"accumulate\": \"f32\", "
                 "\"gemm\": \"unsupported\", \"conv\": \"NHWC x [OC][kH][kW][IC]; IC a multiple of 8, the input under a block in LDS\"}",
                 BLOCK_ROWS, BLOCK_COLS, WAVE_ROWS, WAVE_COLS, KT, K_GROUPS, NTHREADS);
        done = true;
    }
    return buf;
}

inline size_t workspace_bytes(int, int, int) { return 0; }
inline size_t conv_workspace_bytes(int, int, int, int, int, int, int, int, int) { return 0; }

inline int gemm(const void*, const void*, void*, int, int, int, int, int, int, void*, size_t, hipStream_t) {
    return HELIX_ERR_UNSUPPORTED;
}

inline void bench_layout(int M, int N, int K, size_t* ae, size_t* be, size_t* ce, int* lda, int* ldb, int* ldc) {
    *ae = (size_t)M * K; *be = (size_t)N * K; *ce = (size_t)M * N;
    *lda = K; *ldb = K; *ldc = N;
}

// Staged rows under `pixels` consecutive output pixels from a multiple of them, at most: their own, the filter's, and where
// an image ends between them the rows that the next one starts over with.
inline long long staged_rows(int OH, int OW, int kH, int stride, long long pixels) {
    long long rows, crossings;
    if (pixels % OW == 0) {
        rows = pixels / OW;
        crossings = rows % OH == 0 ? rows / OH - 1 : OH % rows == 0 ? 0 : (rows - 2) / OH + 1;
    } else {
        rows = (pixels - 2) / OW + 2;                    // (16 pixels or more)
        crossings = (rows - 2) / OH + 1;
    }
    return (rows - 1) * stride + kH + crossings * (kH > stride ? kH - stride : 0);
}

// Launch parameters of a layer; false where it is not for this configuration (LDS, index ranges).
inline bool make_plan(Params& p, int* lds_bytes, int batch, int H, int W, int IC, int OC, int kH, int kW, int stride, int pad) {
    const int OH = (H + 2 * pad - kH) / stride + 1, OW = (W + 2 * pad - kW) / stride + 1;
    const long long K = (long long)kH * kW * IC, M = (long long)batch * OH * OW;
    const long long x_bytes = (long long)batch * H * W * IC * 2, w_bytes = (long long)OC * K * 2;
    // buffers below the offset that reads zeros, and the 24-bit factors of the kernel's products: rows, row bytes, pixels
    if (IC % 8 != 0 || K * 2 > 0x1000000 || x_bytes >= OOB || w_bytes >= OOB) return false;
    if (M > 0x7fffff || (long long)W * IC * 2 > 0x7fffff || (long long)batch * H > 0x7fffff) return false;
    p.H = H; p.W = W; p.OH = OH; p.OC = OC; p.stride = stride; p.pad = pad; p.M = (int)M; p.kW = kW;
    p.group = IC / 8; p.chunks = (int)(K / 8);
    p.ktiles = (p.chunks + KT_CHUNKS - 1) / KT_CHUNKS; p.tiles_per_part = (p.ktiles + K_GROUPS - 1) / K_GROUPS;
    p.channel_blocks = (OC + BLOCK_COLS - 1) / BLOCK_COLS;
    const long long blocks = (M + BLOCK_ROWS - 1) / BLOCK_ROWS * p.channel_blocks;
    const long long image_rows = (long long)(OH - 1) * stride + kH, row_pixels = (long long)(OW - 1) * stride + kW;
    if (blocks > 0x3fffffff || batch * image_rows > 0x7fffff || row_pixels > LDS_MAX) return false;
    p.blocks = (int)blocks; p.blocks_per_xcd = (p.blocks + NUM_XCD - 1) / NUM_XCD;
    p.image_rows = (int)image_rows; p.row_pixels = (int)row_pixels;
    p.real_pixels = p.row_pixels - pad < W ? p.row_pixels - pad : W;
    if (p.real_pixels < 1) return false;
    // consecutive output pixels twice an odd number of chunks apart (see pixel_of), as close to that as it gets where the
    // stride is even; one chunk behind the channels where K has a remainder to read there
    const int used = p.group + (p.chunks % KT_CHUNKS ? 1 : 0);
    p.pixel_bytes = 16 * (stride % 2 ? used + (6 - used % 4) % 4 : used | 1);
    const long long row_bytes = row_pixels * p.pixel_bytes;
    const long long patch_offset = NWAVES * OWN_BYTES + KT_CHUNKS * ((long long)p.ktiles + 1) * 4;
    const long long patch = staged_rows(OH, OW, kH, stride, BLOCK_ROWS < M ? BLOCK_ROWS : M) * row_bytes;
    const long long lds = patch_offset + patch > SUM_BYTES ? patch_offset + patch : SUM_BYTES;
    if (lds > LDS_MAX) return false;
    p.row_bytes = (int)row_bytes; p.patch_offset = (int)patch_offset;
    p.row_chunks = p.real_pixels * p.group;
    p.x_bytes = (unsigned)x_bytes; p.w_bytes = (unsigned)w_bytes;
    const int border = (p.row_pixels - p.real_pixels) * p.group;
    p.by_OW = helix_fastdiv::make(OW);
    p.by_OH = helix_fastdiv::make(OH);
    p.by_group = helix_fastdiv::make(p.group);
    p.by_kW = helix_fastdiv::make(kW);
    p.by_row_chunks = helix_fastdiv::make(p.row_chunks);
    p.by_image_rows = helix_fastdiv::make(p.image_rows);
    p.by_channel_blocks = helix_fastdiv::make(p.channel_blocks);
    p.by_border = helix_fastdiv::make(border > 0 ? border : 1);
    *lds_bytes = (int)lds;
    return true;
}

inline int conv2d(const void* x, const void* w, void* y, int batch, int H, int W, int IC, int OC, int kH, int kW, int stride,
                  int pad, void*, size_t, hipStream_t s) {
    if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)y & 1)) return HELIX_ERR_INVALID_VALUE;
    Params p{};
    int lds_bytes;
    if (!make_plan(p, &lds_bytes, batch, H, W, IC, OC, kH, kW, stride, pad)) return HELIX_ERR_UNSUPPORTED;
    p.x = (const _Float16*)x; p.w = (const _Float16*)w; p.y = (_Float16*)y;
    constexpr int STORE = TN == 1 ? 4 : 8;     // channels of a lane's store
    p.wide = OC % STORE == 0 && ((uintptr_t)y & (2 * STORE - 1)) == 0;
    static int rc = (int)hipFuncSetAttribute((const void*)helix_conv_patch_f16_kernel<>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX);
    if (rc) return rc;
    hipLaunchKernelGGL(helix_conv_patch_f16_kernel<>, dim3((unsigned)(NUM_XCD * p.blocks_per_xcd)), dim3(NTHREADS), lds_bytes, s, p);
    return (int)hipGetLastError();
}

}  // namespace tpl

#define HELIX_TPL_SCRATCH_BYTES 256   // this family never asks for a workspace
#include "helix_host.h"
