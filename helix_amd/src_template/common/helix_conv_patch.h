// MI355X (gfx950 / CDNA4) convolution template whose input stays in LDS while the filter walks over it, FP16 (PATCH_F32 0) or
// FP32 (PATCH_F32 1).
//
//   y[B,OH,OW,OC] = conv2d(x[B,H,W,IC], w[OC,kH,kW,IC]).  FP16: IC a multiple of 8, FP32 accumulate (MFMA), FP16 out.
//   FP32: any IC, FP32 MFMA.
//
// Role in the reference: the im2col.cu + gemm.cu pair (src_template/Ampere_FP16/im2col.cu:38-97), as the implicit GEMM of
// gemm.hip; this family is for the layers that one is slow on.
//
// What bounds those: gemm.hip gathers a tile's rows from L2 again for every filter tap, and a compute unit takes 46 bytes per
// clock from there, so that a 64 x 64 tile is fed in 2.8 times the time it multiplies; and a layer of few output tiles and
// long K has to be cut along K over workgroups, whose sums meet in a tail of 3.3 us.  Here
//   * a workgroup stages the input rows under its BLOCK_ROWS output pixels in LDS once, with all channels and with the
//     padding, and every tap of the filter reads them there: 16 pixels x 32 channels of one tap are the MFMA's operand, at
//     an LDS offset from each pixel's corner that a table holds (K in chunks of 16 bytes, any number of them; 16 channels, one
//     of each chunk for each of four 16x16x4 products, in FP32, where a last chunk of a pixel may be one of less than four);
//   * K_GROUPS waves share each output tile, each with its part of K, and add their sums through LDS, in order: the few
//     workgroups of a small layer keep their compute units busy, without a second pass over memory;
//   * a wave loads its weights by itself, AHEAD K tiles in front of their use, in rows of 128 bytes, and brings them into the
//     MFMA's order through a piece of LDS that is its own: no barrier between the first product and the last.  (Loaded in the
//     MFMA's order, 16 rows x 64 bytes per instruction, they come at a quarter of the rate: 15.7 instead of 53 bytes per clock
//     and CU, one cache line looked up for each lane.)
//   * results leave from registers, 16 bytes per lane;
//   * FP32 sums are cut as common/helix_sums.h says: few results as exactly as sgemm.hip's K groups (1.1e-7 in the norm at 2 x 128 x 7 x 7
//     3x3 -> 96, where a chain per part of K left 2.3e-7), many in chains of 256 (2.8e-7 at 32 x 128 x 28 x 28, 6.0e-7 in one).
//
// Measured (us per launch, the fastest configuration of the implicit GEMM / of this family; batch x channels x image, filter):
//   FP16  4 x 256 x 14 x 14 3x3 -> 256 10.1 / 6.6    2 x 512 x 16 x 16 3x3 -> 256 10.1 / 6.5    2 x 112 x 14 x 14 3x3 -> 208 7.4 / 4.7
//         1 x 256 x 13 x 13 3x3 -> 160 7.7 / 5.0     2 x 96 x 15 x 15 5x5 -> 512 9.4 / 6.6      4 x 192 x 9 x 9 3x3 -> 48 6.7 / 4.6
//         32 x 64 x 56 x 56 3x3 -> 64 15.1 / 14.5    32 x 256 x 14 x 14 3x3 -> 256 15.2 / 13.5  16 x 48 x 40 x 40 5x5 -> 96 13.0 / 11.3
//   FP32  32 x 128 x 28 x 28 3x3 -> 128 69.3 / 67.7  4 x 256 x 14 x 14 3x3 -> 256 18.8 / 17.2   5 x 32 x 64 x 64 5x5 -> 64 27.3 / 23.5
//         1 x 24 x 10 x 10 3x3 -> 256 7.3 / 4.5      2 x 128 x 7 x 7 3x3 -> 96 9.0 / 5.9        2 x 25 x 70 x 70 1x1 -> 16 8.5 / 5.0
//         22 x 3 x 154 x 154 5x5 stride 4 -> 64 21.1 / 13.4, 2 x 3 x 122 x 122 5x5 stride 2 -> 32 9.1 / 6.0
// Slower, and left to the implicit GEMM by the selection, which times both: FP16 filters with stride 2 on large images; images or
// channel counts that leave room for few pixels in LDS (FP16 9 x 96 x 106 x 106 3x3 -> 128 32 / 50).  Strips of columns and passes
// over the channels, which would fit those, were built in FP16 and measured: never ahead there, half a microsecond slower
// everywhere else.  What bounds it where it runs: small layers launch, first loads and staging (2.6 + 2 us); large FP16 ones LDS (22
// KB read and written per 28 products of a 112 x 32 wave tile), with staging and stores in front of and behind the loop over K, not
// beside it; FP32 ones the matrix pipes, at 0.75 of their rate.
//
// Compile-time parameters (-D, one shared library per combination):
//   BLOCK_ROWS x BLOCK_COLS   output pixels x channels of a workgroup
//   WAVE_ROWS  x WAVE_COLS    of a wave, multiples of 16
//   K_GROUPS                  parts of K, each on its own wave
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <type_traits>

#include "helix_abi.h"
#include "helix_fastdiv.h"
#include "helix_sums.h"

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
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx3 __attribute__((ext_vector_type(3)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));

constexpr bool F32 = PATCH_F32;
typedef std::conditional<F32, float, _Float16>::type elem;
constexpr int EB = sizeof(elem), CE = 16 / EB;                   // bytes of an element, elements of a 16-byte chunk

constexpr int TM = WAVE_ROWS / 16, TN = WAVE_COLS / 16;          // MFMA tiles of a wave
constexpr int WAVES_M = BLOCK_ROWS / WAVE_ROWS, WAVES_N = BLOCK_COLS / WAVE_COLS;
constexpr int NWAVES = WAVES_M * WAVES_N * K_GROUPS, NTHREADS = 64 * NWAVES;
constexpr int KT_CHUNKS = 8, KT_BYTES = 128;  // K tile: what a wave loads of its weights at a time, two steps of four chunks
constexpr int PRODUCTS = F32 ? 4 : 1;         // MFMAs of a step and tile: one 16x16x32, or 16x16x4 ones of one element of each chunk
constexpr int AHEAD = 2;                      // K tiles of weights in flight in registers
constexpr int OWN_BYTES = WAVE_COLS * KT_BYTES; // a wave's piece of LDS for its weights
constexpr int ZERO_BYTES = 16;                // in front of everything in LDS: what the K chunks of a last tile beyond the filter read,
constexpr int BEYOND = -(1 << 24);            // at this offset from any pixel (REST, see table_entry and operand_at)
constexpr int TABLE_OFFSET = ZERO_BYTES + NWAVES * OWN_BYTES;   // LDS offsets of the K chunks from a pixel's corner
constexpr int SUM_BYTES = K_GROUPS > 1 ? NWAVES * TM * TN * 1024 : 0;
constexpr int LDS_MAX = 160 * 1024;
constexpr int NUM_XCD = 8;
constexpr unsigned OOB = 0x40000000u;         // byte offset beyond any buffer (they stay below it), twice too: the load returns zeros

static_assert(BLOCK_ROWS % WAVE_ROWS == 0 && BLOCK_COLS % WAVE_COLS == 0 && WAVE_ROWS % 16 == 0 && WAVE_COLS % 16 == 0, "tiles");
static_assert(F32 || TN == 1 || TN % 2 == 0, "a lane's halves are four channels of a single tile or eight of a pair");
static_assert(NTHREADS <= 512 && SUM_BYTES <= LDS_MAX, "workgroup");

struct Params {
    const elem* x;   // NHWC
    const elem* w;   // [OC][kH][kW][IC]
    elem* y;             // NHWC
    int H, W, OH, OC, stride, pad, kW;
    int M;                                 // output pixels of the batch
    int group, tail;                       // 16-byte chunks of a pixel's channels, and elements of a last one that is not whole
    int channel_bytes;                     // of a pixel
    int taps, chunks, ktiles, tiles_per_part;   // filter taps, K in 16-byte chunks, in tiles of eight, and the tiles of one wave's part
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
__device__ __forceinline__ uintx4 load16(__amdgpu_buffer_rsrc_t r, unsigned at) {
    return __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)at, 0, 0));
}

// n / d: the bits of FastDiv::div through the high word of one 32-bit product, which the staging loop's three divisions a chunk
// are a third of.
__host__ __device__ __forceinline__ int quotient(const FastDiv& d, int n) {
    return (int)((unsigned)((unsigned long long)((unsigned)n << 1) * d.mul >> 32) >> (d.shift - 31));
}

// A product of two 24-bit factors
__host__ __device__ __forceinline__ int times(int a, int b) {
#ifdef __HIP_DEVICE_COMPILE__
    return __mul24(a, b);
#else
    return a * b;
#endif
}

// LDS offset of K chunk j from a pixel's corner; the table holds those of the K tiles and of one more, which is read ahead (by a wave
// whose part of K is empty, too) and not multiplied.  Beyond the filter it is the zeros' where a tile has such chunks (REST), else
// all of them are read ahead only and take the pixel's first chunk, which is a place inside the patch.
template <bool REST>
__host__ __device__ __forceinline__ int table_entry(const Params& p, int j) {
    const int tap = quotient(p.by_group, j), g = j - times(tap, p.group);
    const int kh = quotient(p.by_kW, tap), kw = tap - times(kh, p.kW);
    return j < p.chunks ? times(kh, p.row_bytes) + times(kw, p.pixel_bytes) + g * 16 : REST ? BEYOND : 0;
}

// LDS offset of that chunk of the pixel whose corner is at `at`
template <bool REST>
__host__ __device__ __forceinline__ int operand_at(int at, int o) { return !REST || at + o > 0 ? at + o : 0; }

// One chunk of a pixel or of a filter tap.  TAIL (FP32, where an element is a dword): `elements` of it, and not a byte beyond
// them, which may be the buffer's end.  (No branch on that: one inside the loop over K made every load wait for itself.)
template <bool TAIL>
__device__ __forceinline__ uintx4 load_chunk(__amdgpu_buffer_rsrc_t r, unsigned at, int elements) {
    if constexpr (!TAIL) return load16(r, at);
    uintx4 v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)(e < elements ? at + 4 * e : OOB), 0, 0);
    return v;
}

// Output channel (within a wave's) of row r of MFMA tile j: two tiles leave a lane of quarter q with the channels
// 8 q .. 8 q + 7 of their 32, a single one with 4 q .. 4 q + 3 of its 16.
__device__ __forceinline__ int channel_of(int j, int r) {
    return F32 || TN % 2 ? j * 16 + r : (j >> 1) * 32 + (r >> 2) * 8 + (j & 1) * 4 + (r & 3);
}

// Pixel (within an MFMA tile) of lane l.  ds_read_b128 serves lanes {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same of the
// upper half together.
__device__ __forceinline__ int pixel_of(int r) { return r < 4 ? r : r < 12 ? r + 4 : r - 8; }

// (REST: K is not whole tiles.  The tile parameters are template arguments for the symbol name's sake: a profiler lists configurations separately)
// (wave tiles of more than ten have no room for two sets of FP32 accumulators in 256 registers; one of their workgroups fills a CU)
template <bool TAIL, bool REST, int SUMS, int T_BM = BLOCK_ROWS, int T_BN = BLOCK_COLS, int T_WM = WAVE_ROWS, int T_WN = WAVE_COLS, int T_KG = K_GROUPS, bool T_F32 = F32>
__global__ __launch_bounds__(NTHREADS, F32 && TM * TN > 10 ? 1 : 2) void helix_conv_patch_kernel(const Params p) {
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
    unsigned w_at[2 * TN];               // 8 rows of a tile at a time: lane l takes chunk l % 8 of row l / 8
#pragma unroll
    for (int d = 0; d < 2 * TN; d++) {
        const int n = oc0 + channel_of(d >> 1, (d & 1) * 8 + (lane >> 3));
        w_at[d] = n < p.OC ? (unsigned)(n * (p.taps * p.channel_bytes)) : OOB;
    }
    struct At { unsigned offset; int elements; };
    auto tile_at = [&](int t) -> At {
        const int c = KT_CHUNKS * t + (lane & 7);
        if (!TAIL) return At{c < chunk_end ? (unsigned)c * 16 : OOB, 4};
        const int tap = quotient(p.by_group, c), g = c - __mul24(tap, p.group);
        return At{c < chunk_end ? (unsigned)(__mul24(tap, p.channel_bytes) + g * 16) : OOB, g == p.group - 1 ? p.tail : 4};
    };
    uintx4 st[AHEAD][2 * TN];
#pragma unroll
    for (int u = 0; u < AHEAD; u++) {
        const At k = tile_at(t_begin + u);
#pragma unroll
        for (int d = 0; d < 2 * TN; d++) st[u][d] = load_chunk<TAIL>(rw, w_at[d] + k.offset, k.elements);
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
        const int total = rows * p.row_chunks, gap = p.pixel_bytes - p.group * 16, image_row_bytes = p.W * p.channel_bytes;
        constexpr int BATCH = 8;                            // loads of a thread in flight
        for (int i0 = tid; i0 < total; i0 += NTHREADS * BATCH) {
            uintx4 v[BATCH];
            int dst[BATCH];
#pragma unroll
            for (int u = 0; u < BATCH; u++) {
                const int i = i0 + u * NTHREADS;
                const int row = quotient(p.by_row_chunks, i), c = i - __mul24(row, p.row_chunks);
                const int image = quotient(p.by_image_rows, row0 + row), ih = row0 + row - __mul24(image, p.image_rows) - p.pad;
                const int px = quotient(p.by_group, c), g = c - __mul24(px, p.group);
                const bool inside = (i < total) & ((unsigned)ih < (unsigned)p.H);
                const int in_row = TAIL ? __mul24(px, p.channel_bytes) + g * 16 : c * 16;
                v[u] = load_chunk<TAIL>(rx, inside ? (unsigned)(__mul24(__mul24(image, p.H) + ih, image_row_bytes) + in_row) : OOB, g == p.group - 1 ? p.tail : 4);
                dst[u] = i < total ? __mul24(row, p.row_bytes) + c * 16 + __mul24(px, gap) : -1;
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
        if (tid == 0) *(uintx4*)smem = uintx4{0, 0, 0, 0};
        // LDS offset of each K chunk from a pixel's corner
        for (int j = tid; j < KT_CHUNKS * (p.ktiles + 1); j += NTHREADS) ((int*)(smem + TABLE_OFFSET))[j] = table_entry<REST>(p, j);
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
    helix_sums::Sums<TM, TN, SUMS> sums;
    sums.start();
    const int* table = (const int*)(smem + TABLE_OFFSET) + q;
    typedef std::conditional<F32, floatx4, half8>::type frag;
    // rows of 128 bytes, 16-byte chunk c of row r at c ^ (r / 2 mod 8): reads and writes free of bank conflicts
    unsigned char* own = smem + ZERO_BYTES + wave * OWN_BYTES;
    unsigned char* own_write = own + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 4)) << 4);
    unsigned char* own_write_odd = own + (lane >> 3) * 128 + (((lane & 7) ^ ((lane >> 4) + 4)) << 4);
    auto write_b = [&](int d, uintx4 v) { *(uintx4*)((d & 1 ? own_write_odd : own_write) + d * 1024) = v; };
    auto read_b = [&](int s, int j) -> frag { return *(const frag*)(own + j * 2048 + r * 128 + (((s * 4 + q) ^ (r >> 1)) << 4)); };
    frag a[2][TM], b[2][TN];
    int off[2];
    constexpr int SLOTS = TM * TN * PRODUCTS;
    auto multiply = [&](int g, int s) {
        const int i = g % TM, j = g / TM % TN, e = g / (TM * TN);
        if constexpr (F32) sums.multiply(i, j, s * PRODUCTS + e, b[s][j][e], a[s][i][e]);
        else sums.sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[s][j], a[s][i], sums.sum[i][j], 0, 0, 0);
    };
    // One K tile, st holding the weights of the next one.  Behind each MFMA its share of the other instructions, in the order in
    // which the products take them and in the first two thirds of the step, so that the last ones have arrived when the next
    // step begins: the reads of the second step's operands behind the first step's products, of the next tile's first step's
    // behind the second step's, once its weights have taken this tile's place (a wave's LDS instructions execute in their
    // order); then the loads AHEAD tiles on.  off[s]: LDS offset of the chunks that are read behind step s.
    auto read_operand = [&](int e, int s, int o) {          // weights of the first 16 channels, pixels, other weights
        if (e == 0) b[s][0] = read_b(s, 0);
        else if (e <= TM) a[s][e - 1] = *(const frag*)(smem + operand_at<REST>(at[e - 1], o));
        else b[s][e - TM] = read_b(s, e - TM);
    };
    constexpr int W = 2 * TN, EARLY = 2 * SLOTS / 3 > 0 ? 2 * SLOTS / 3 : 1;
    auto tile = [&](int t, uintx4 (&stv)[W]) {
        const At k = tile_at(t + 1 + AHEAD);
#pragma unroll
        for (int g = 0; g < SLOTS; g++) {
            multiply(g, 0);
            constexpr int COUNT = 1 + TM + TN;
#pragma unroll
            for (int e = 0; e < COUNT; e++) {
                if (e * EARLY / COUNT != g) continue;
                if (e == 0) off[1] = table[KT_CHUNKS * (t + 1)];
                else read_operand(e - 1, 1, off[0]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int g = 0; g < SLOTS; g++) {
            multiply(g, 1);
            constexpr int COUNT = 1 + W + TM + TN;
#pragma unroll
            for (int e = 0; e < COUNT; e++) {
                if (e * EARLY / COUNT != g) continue;
                if (e == 0) off[0] = table[KT_CHUNKS * (t + 1) + 4];
                else if (e <= W) write_b(e - 1, stv[e - 1]);
                else read_operand(e - 1 - W, 0, off[1]);
            }
#pragma unroll
            for (int d = 0; d < W; d++)
                if (EARLY - 1 + d * (SLOTS - EARLY + 1) / W == g) stv[d] = load_chunk<TAIL>(rw, w_at[d] + k.offset, k.elements);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // the first tile's operands; its registers take tile AHEAD
    {
        const At k = tile_at(t_begin + AHEAD);
#pragma unroll
        for (int d = 0; d < 2 * TN; d++) {
            write_b(d, st[0][d]);
            st[0][d] = load_chunk<TAIL>(rw, w_at[d] + k.offset, k.elements);
        }
        const int o = table[KT_CHUNKS * t_begin];
#pragma unroll
        for (int e = 0; e < TM + TN; e++) read_operand(e, 0, o);
        off[0] = table[KT_CHUNKS * t_begin + 4];
    }
    // a last tile of one step only
    const bool half = REST && chunk_end > KT_CHUNKS * t_begin && (chunk_end - 1) % KT_CHUNKS < 4;
    const int t_whole = t_end - half;
    int t = t_begin;
    if constexpr (sums.BLOCK_TILES == 0) {
        for (; t + AHEAD <= t_whole; t += AHEAD) {
            tile(t, st[1]);
            tile(t + 1, st[0]);
        }
    } else {
        constexpr int BLOCK_TILES = sums.BLOCK_TILES;
        static_assert(BLOCK_TILES == 1 || BLOCK_TILES % AHEAD == 0, "blocks of sums end between tiles");
        for (int end; t + AHEAD <= t_whole; ) {
            end = BLOCK_TILES == 1 || BLOCK_TILES > t_whole - t ? t + (t_whole - t) / AHEAD * AHEAD : t + BLOCK_TILES;
            for (; t < end; t += AHEAD) {
                tile(t, st[1]);
                if constexpr (BLOCK_TILES == 1) sums.end_block();
                tile(t + 1, st[0]);
                if constexpr (BLOCK_TILES == 1) sums.end_block();
            }
            if (BLOCK_TILES > 1 && (t < t_whole || half)) sums.end_block();
        }
    }
    if (t < t_whole) {
        tile(t, st[1]);
        if constexpr (sums.BLOCK_TILES == 1) sums.end_block();
    }
    if (half)
#pragma unroll
        for (int g = 0; g < SLOTS; g++) multiply(g, 0);
    sums.finish(half);

    // ---- results -----------------------------------------------------------------------------------------------------
    constexpr int PAIR = F32 || TN % 2 ? 1 : 2, UNITS = TM * (TN / PAIR);
    auto store = [&](int i, int jj, const floatx4 (&v)[PAIR]) {
        const int m = m0 + (wave_m * TM + i) * 16 + pixel_of(r);
        if (m > m_last) return;
        const int n = oc0 + jj * (16 * PAIR) + q * (4 * PAIR);
        elem* dst = p.y + (size_t)m * p.OC + n;
        typedef elem results __attribute__((ext_vector_type(4 * PAIR)));
        results h;
#pragma unroll
        for (int e = 0; e < 4 * PAIR; e++) h[e] = (elem)v[e >> 2][e & 3];
        if (p.wide) {
            if (n < p.OC) *(results*)dst = h;
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
                for (int e = 0; e < PAIR; e++) v[e] = sums.sum[i][jj * PAIR + e];
                store(i, jj, v);
            }
    } else {
        // parts of K: added through LDS in their order, the units of a wave's tile shared out over its parts
        __syncthreads();
        floatx4* parts = (floatx4*)smem + (size_t)(wave_m * WAVES_N + wave_n) * K_GROUPS * (TM * TN * 64);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) parts[(part * (TM * TN) + i * TN + j) * 64 + lane] = sums.sum[i][j];
        __syncthreads();
        for (int u = part; u < UNITS; u += K_GROUPS) {
            const int i = u / (TN / PAIR), jj = u % (TN / PAIR);
            floatx4 v[PAIR];
#pragma unroll
            for (int e = 0; e < PAIR; e++) v[e] = parts[(i * TN + jj * PAIR + e) * 64 + lane];
            for (int k = 1; k < K_GROUPS; k++)
#pragma unroll
                for (int e = 0; e < PAIR; e++) v[e] += parts[(k * (TM * TN) + i * TN + jj * PAIR + e) * 64 + lane];
            store(i, jj, v);
        }
    }
}
}  // namespace

// -------------------------------------------------------------------------------------------------
// host side
// -------------------------------------------------------------------------------------------------
namespace tpl {

constexpr int kElemBytes = EB;

inline const char* info_json() {
    static char buf[1024];
    static bool done = false;
    if (!done) {
        snprintf(buf, sizeof(buf),
                 "{\"family\": \"%s\", \"input_in_lds\": 1, \"arch\": \"gfx950\", \"mfma\": \"%s\", "
                 "\"block_rows\": %d, \"block_cols\": %d, \"wave_rows\": %d, \"wave_cols\": %d, \"block_k\": %d, "
                 "\"k_groups\": %d, \"split_k\": 1, \"threads\": %d, \"accumulate\": \"f32\", "
                 "\"gemm\": \"unsupported\", \"conv\": \"NHWC x [OC][kH][kW][IC]; the input under a block in LDS; %s\"}",
                 F32 ? "sgemm_f32" : "gemm_f16", F32 ? "v_mfma_f32_16x16x4_f32" : "v_mfma_f32_16x16x32_f16", BLOCK_ROWS, BLOCK_COLS,
                 WAVE_ROWS, WAVE_COLS, KT_BYTES / EB, K_GROUPS, NTHREADS, F32 ? "any IC" : "IC a multiple of 8");
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
    const long long M = (long long)batch * OH * OW, pixel = (long long)IC * EB, filter = (long long)kH * kW * pixel;
    const long long x_bytes = (long long)batch * H * W * pixel, w_bytes = (long long)OC * filter;
    // (16-bit elements: chunks whole; FP32: any channel count, see load_chunk.)  Buffers below the offset that reads zeros, and
    // the 24-bit factors of the kernel's products: rows, row bytes, pixels
    if ((!F32 && IC % CE != 0) || filter > 0x1000000 || x_bytes >= OOB || w_bytes >= OOB) return false;
    if (M > 0x7fffff || W * pixel > 0x7fffff || (long long)batch * H > 0x7fffff) return false;
    p.H = H; p.W = W; p.OH = OH; p.OC = OC; p.stride = stride; p.pad = pad; p.M = (int)M; p.kW = kW;
    p.group = (IC + CE - 1) / CE; p.tail = IC % CE; p.channel_bytes = (int)pixel;
    p.taps = kH * kW; p.chunks = p.taps * p.group;
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
    // stride is even
    p.pixel_bytes = 16 * (stride % 2 ? p.group + (6 - p.group % 4) % 4 : p.group | 1);
    const long long row_bytes = row_pixels * p.pixel_bytes;
    const long long patch_offset = TABLE_OFFSET + KT_CHUNKS * ((long long)p.ktiles + 1) * 4;
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

// Which variant runs a layer: REST of the kernel
inline bool has_rest(const Params& p) { return (F32 && p.tail) || p.chunks % KT_CHUNKS; }

template <bool TAIL, bool REST, int SUMS>
inline int launch(const Params& p, int lds_bytes, hipStream_t s) {
    static int rc = (int)hipFuncSetAttribute((const void*)helix_conv_patch_kernel<TAIL, REST, SUMS>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX);
    if (rc) return rc;
    hipLaunchKernelGGL((helix_conv_patch_kernel<TAIL, REST, SUMS>), dim3((unsigned)(NUM_XCD * p.blocks_per_xcd)), dim3(NTHREADS), lds_bytes, s, p);
    return (int)hipGetLastError();
}

template <int SUMS>
inline int launch_variant(const Params& p, int lds_bytes, hipStream_t s) {
    // (with a tail the compiler holds the accumulators of HALVES twice)
    if constexpr (F32)
        if (p.tail) return launch<true, true, SUMS == helix_sums::HALVES && TM * TN >= 8 ? helix_sums::TILES : SUMS>(p, lds_bytes, s);
    return has_rest(p) ? launch<false, true, SUMS>(p, lds_bytes, s) : launch<false, false, SUMS>(p, lds_bytes, s);
}

inline int conv2d(const void* x, const void* w, void* y, int batch, int H, int W, int IC, int OC, int kH, int kW, int stride,
                  int pad, void*, size_t, hipStream_t s) {
    if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)y & (EB - 1))) return HELIX_ERR_INVALID_VALUE;
    Params p{};
    int lds_bytes;
    if (!make_plan(p, &lds_bytes, batch, H, W, IC, OC, kH, kW, stride, pad)) return HELIX_ERR_UNSUPPORTED;
    p.x = (const elem*)x; p.w = (const elem*)w; p.y = (elem*)y;
    constexpr int STORE = F32 || TN == 1 ? 4 : 8;      // channels of a lane's store
    p.wide = OC % STORE == 0 && ((uintptr_t)y & (EB * STORE - 1)) == 0;
    if constexpr (F32) {
        switch (helix_sums::mode_of(p.M, OC, (long long)p.taps * IC, K_GROUPS)) {
            case helix_sums::FINE: return launch_variant<helix_sums::finest(TM, TN)>(p, lds_bytes, s);
            case helix_sums::HALVES: return launch_variant<helix_sums::HALVES>(p, lds_bytes, s);
            default: return launch_variant<helix_sums::BLOCKS>(p, lds_bytes, s);
        }
    } else {
        return launch_variant<helix_sums::CHAIN>(p, lds_bytes, s);
    }
}

}  // namespace tpl

#define HELIX_TPL_SCRATCH_BYTES 256   // this family never asks for a workspace
#include "helix_host.h"
