// FP16 convolution of thin inputs: one to four channels, the first layers of CNNs (3 -> 64, 7x7 stride 2) and of
// speech models (1 -> 32, 5x20 stride 2).  Used by the FP16 tile libraries' helix_conv2d for such layers, whatever
// their tile parameters are, where it is the faster path (is_faster below).
//
// What bounds such a layer is its output (batch 32, 224 x 224 x 3 -> 64, 7x7 stride 2: 51 MB written, 9.6 MB read, 7.6
// Gflop): the general path copied the activations to eight channels and walked K = kH * kW * 8, 2.7 times the products,
// gathering every tile's rows again for each K tile.  Here a workgroup
//   * takes a block of output rows and columns of one image (whole rows unless they are few and wide) and 64 output
//     channels, and further such blocks while there are more of them than workgroups the chip holds;
//   * stages the input rows under the block in LDS once, four halves per pixel (missing channels zero), columns of padding
//     included, so that the two pixels x four channels that an MFMA lane supplies are 16 consecutive bytes of LDS at
//     a fixed distance from its output pixel's corner: no index arithmetic per tap;
//   * walks K in chunks of (filter row, pair of filter columns): four chunks make one 32-wide MFMA step, so a 7x7 filter
//     is 7 steps (K = 224 where 147 is the least) and a 3x3 filter 2 (64 / 27);
//   * keeps the weights of all steps in registers (up to 7 steps: 112 registers) and reads each 16-pixel fragment
//     once for the 64 channels (KS > 0), or, for longer filters, reads both operands from LDS (KS = 0);
//   * holds the channels of an MFMA tile in such an order that a lane ends up with eight consecutive channels: results
//     go out 16 bytes per lane, 64 contiguous bytes per pixel and instruction, without passing through LDS.  Plain
//     stores: the L2 joins the two halves of a pixel's 128 bytes (non-temporal ones took the 3x3 layer 67 us).
// A pair that hangs over the end of a filter row takes its second pixel as zero, and chunks beyond the filter read a
// zeroed slot: exactly the filter's taps contribute, whatever the neighbouring pixels hold.
//
// Measured, us per launch (helix_bench_conv), the general path's fastest configuration against this one: batch 32, 224 x 224
// x 3 -> 64: 7x7 stride 2 58 / 22, 3x3 88 / 36 (5.9 TB/s), 11x11 stride 4 -> 96 49 / 28; batch 20, 180 x 180 x 3, 5x5 51 / 21;
// batch 1, 7x7 10.2 / 6.4, 3x3 10.4 / 6.5; 4 x 161 x 700 x 1 -> 32, 5x20 stride 2 33 / 14.  The weights' fragments are packed from
// four dwords each with all of a thread's loads in flight; half by half out of LDS before, on the same memory in turn, one set of
// operands and three: 7x7 at batch 32 21.2 / 21.0 and 21.2 / 20.8 (single rounds 20.4 - 23), at batch 1 6.7 / 6.45, 11x11 31.5 / 30.8 and
// 32.5 / 31.6, at batch 1 11.0 / 10.0; 3x3 36.1 / 36.1 and 46.2 / 46.7.  Two cards put the 7x7 layer at 19.7 and 21.5.
// What is left of it: 2.5 us of launch, about 5 us until weights and patch are in place (all workgroups start together, so nothing
// overlaps it), then 51 MB of results at some 3.7 TB/s, where 5.7 would take 9 us; what holds these up has not been found.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "helix_abi.h"
#include "helix_fastdiv.h"

namespace helix_conv_thin {
namespace {   // internal linkage: every library carries its own copy and exports none of it

using helix_fastdiv::FastDiv;
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx3 __attribute__((ext_vector_type(3)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));

constexpr int OC_BLOCK = 64;                        // output channels of a workgroup, in 16-wide MFMA tiles (96 for some layers, see make_plan)
constexpr int step_bytes(int nt) { return nt * 64 * 16; }      // packed weights of one MFMA step
constexpr int ZERO_BYTES = 16;                      // a zeroed slot in front of the patch
constexpr int LDS_MAX = 160 * 1024;
constexpr int MAX_STEPS = 24;
constexpr int OOB = 0x7fffffff;                     // byte offset beyond any buffer: the load returns zeros
constexpr int threads_of(int ks) { return ks ? 256 : 512; }    // weights in LDS leave room for one workgroup per CU
constexpr int resident_of(int ks, int nt) { return (ks == 7 ? 2 : ks == 4 ? 3 : ks == 0 ? 1 : 4) - (nt == 6); }   // workgroups per CU the registers allow

struct Params {
    const _Float16* x;   // NHWC
    const _Float16* w;   // [OC][kH][kW][IC]
    _Float16* y;         // NHWC
    int H, W, IC, OC, OH, OW, kH, kW, stride, pad;
    int pairs, chunks, steps;      // column pairs per filter row, chunks = kH * pairs, MFMA steps of four chunks
    int rows, cols;                // output rows and columns of a block
    int row_blocks, col_blocks, blocks;   // per image; over the batch
    int patch_rows, patch_cols;    // staged input rows and pixels per row (even)
    int raw_offset, packed_offset; // LDS byte offsets of the weights as they lie and as the MFMAs take them
    int unit_pixels;               // pixels a staging thread moves at once: 4 (three channels) or 1
    unsigned x_bytes;
    FastDiv by_cols, by_row_blocks, by_col_blocks, by_pairs, by_units;   // by_units: units that cover one staged row
};

// Where the 24 bytes of four three-channel pixels at byte `at` of x (the unit) are loaded from: seven whole dwords from byte
// `from` on, never beyond the last whole dword of x.  Near the end of x these start in front of the unit's first dword and are
// moved down by `behind` of them; what then lies behind the end belongs to no pixel of the row.  An odd number of halves leaves
// the last one in no whole dword: it is read by itself and moved in behind the last of them (a unit that holds it is always
// moved, by one dword or more).  x holds at least 28 bytes.
struct Window { int from, behind; };
__host__ __device__ __forceinline__ Window window_of(int at, int x_bytes) {
    const int whole = x_bytes & ~3, first = at & ~3, last = whole - 28;
    const int from = first < last ? first : last;
    return Window{from, (first - from) >> 2};
}

// 16 bytes of LDS at an address that is a multiple of 8
__device__ __forceinline__ uintx4 read16(const unsigned char* p) {
    const uintx2 lo = *(const uintx2*)p, hi = *(const uintx2*)(p + 8);
    return uintx4{lo[0], lo[1], hi[0], hi[1]};
}

// Output channel (within the block) of row r of MFMA tile j: after tiles 2i and 2i + 1 the lanes of quarter q hold
// channels 32 i + 8 q + {0..3} and {4..7} of their pixel.
__device__ __forceinline__ int channel_of(int j, int r) { return (j >> 1) * 32 + (r >> 2) * 8 + (j & 1) * 4 + (r & 3); }

template <int KS, int NT>
__global__ __launch_bounds__(threads_of(KS), resident_of(KS, NT) * threads_of(KS) / 256) void helix_conv_thin_f16_kernel(const Params p) {
    constexpr int THREADS = threads_of(KS), WAVES = THREADS / 64;
    constexpr int STEP_BYTES = step_bytes(NT), CHANNELS = 16 * NT;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int oc0 = (int)blockIdx.y * CHANNELS;
    const int ocs = (p.OC - oc0) < CHANNELS ? (p.OC - oc0) : CHANNELS;

    // ---- input under a block of output pixels: one unit is unit_pixels pixels of one row, from an input column that is a
    // multiple of unit_pixels --------------------------------------------------------------------------------------------
    unsigned char* patch = smem + ZERO_BYTES;
    const int units = p.by_units.d, total_units = p.patch_rows * units;
    struct Block { int image, oh0, ow0; };
    auto block_of = [&](int g) -> Block {
        const int t = p.by_col_blocks.div(g), cb = g - t * p.col_blocks;
        const int image = p.by_row_blocks.div(t);
        return Block{image, (t - image * p.row_blocks) * p.rows, cb * p.cols};
    };
    struct Unit { uintx4 a; uintx2 b; };                       // 24 bytes: four pixels of three channels, or one pixel in a
    auto first_column = [&](int iw) -> int { return p.unit_pixels == 4 ? iw & ~3 : iw; };
    // x as whole dwords (three channels put a pixel at any even byte: the dwords around a unit are shifted into place);
    // an offset beyond the buffer reads zeros
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(p.x), 0, (int)p.x_bytes, 0x00020000);
    auto load_unit = [&](const Block& k, int i) -> Unit {
        Unit v{{0, 0, 0, 0}, {0, 0}};
        const int pr = p.by_units.div(i), u = i - pr * units;
        const int ih = k.oh0 * p.stride - p.pad + pr, iw = first_column(k.ow0 * p.stride - p.pad) + u * p.unit_pixels;
        const bool inside = (i < total_units) & ((unsigned)ih < (unsigned)p.H) & ((unsigned)iw < (unsigned)p.W);
        const int at = (((k.image * p.H + ih) * p.W + iw) * p.IC) * 2;
        if (p.unit_pixels == 4) {
            const Window n = window_of(at, (int)p.x_bytes);
            const uintx4 lo = __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(rx, inside ? n.from : OOB, 0, 0));
            const uintx3 hi = __builtin_bit_cast(uintx3, __builtin_amdgcn_raw_buffer_load_b96(rx, inside ? n.from + 16 : OOB, 0, 0));
            unsigned w[7] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2]};
            for (int behind = inside ? n.behind : 0; __any(behind > 0); behind--) {
#pragma unroll
                for (int e = 0; e < 6; e++) w[e] = behind > 0 ? w[e + 1] : w[e];
                const unsigned half = __builtin_amdgcn_raw_buffer_load_b16(rx, (int)p.x_bytes - 2, 0, 0);
                w[6] = behind > 0 ? half : w[6];
            }
#pragma unroll
            for (int e = 0; e < 4; e++) v.a[e] = __builtin_amdgcn_alignbyte(w[e + 1], w[e], at & 2);
            v.b[0] = __builtin_amdgcn_alignbyte(w[5], w[4], at & 2);
            v.b[1] = __builtin_amdgcn_alignbyte(w[6], w[5], at & 2);
        } else {
            unsigned short e[4] = {0, 0, 0, 0};
#pragma unroll
            for (int c = 0; c < 4; c++)
                if (c < p.IC) e[c] = __builtin_amdgcn_raw_buffer_load_b16(rx, inside ? at + 2 * c : OOB, 0, 0);
            v.a[0] = (unsigned)e[0] | (unsigned)e[1] << 16;
            v.a[1] = (unsigned)e[2] | (unsigned)e[3] << 16;
        }
        return v;
    };
    auto store_unit = [&](const Block& k, int i, const Unit& v) {
        if (i >= total_units) return;
        const int pr = p.by_units.div(i), u = i - pr * units, iw0 = k.ow0 * p.stride - p.pad;
        const int iw = first_column(iw0) + u * p.unit_pixels, pc = iw - iw0;
        unsigned char* dst = patch + (pr * p.patch_cols + pc) * 8;
        auto put = [&](int c, unsigned lo, unsigned hi) {      // a unit may reach past the end of the row
            const bool in = iw + c < p.W;
            if ((unsigned)(pc + c) < (unsigned)p.patch_cols) *(uintx2*)(dst + c * 8) = uintx2{in ? lo : 0u, in ? hi : 0u};
        };
        if (p.unit_pixels == 4) {
            put(0, v.a[0], v.a[1] & 0xffffu);
            put(1, v.a[1] >> 16 | v.a[2] << 16, v.a[2] >> 16);
            put(2, v.a[3], v.b[0] & 0xffffu);
            put(3, v.b[0] >> 16 | v.b[1] << 16, v.b[1] >> 16);
        } else {
            put(0, v.a[0], v.a[1]);
        }
    };
    // ---- weights: as they lie; with more than four steps of them the loads of a thread are all in flight at once (7x7 at
    // batch 32 21.3 -> 20.8 us, at 1 6.66 -> 6.47, 11x11 level; of fewer there is one or two, and the plain loop is the shorter one) -----
    const int taps = p.kH * p.kW, filter = taps * p.IC, halves = ocs * filter;
    const _Float16* src = p.w + (size_t)oc0 * filter;         // a multiple of 32 filters in: 16-byte aligned
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(src), 0, halves * 2, 0x00020000);
    constexpr bool AT_ONCE = KS == 0 || KS > 4;
    constexpr int WF = AT_ONCE ? 6 : 0;
    uintx4 first[WF + 1];
    auto load_weights = [&](int i) -> uintx4 {                 // 16 bytes, where all of them are filters of this block
        return __builtin_bit_cast(uintx4, __builtin_amdgcn_raw_buffer_load_b128(rw, i < halves / 8 ? i * 16 : OOB, 0, 0));
    };

    // the first PF units per thread of a block are requested ahead: the first block's in front of the work on the weights,
    // a later block's in front of the multiplication of the one before it
    constexpr int PF = 4;
    Unit early[PF];
    int g = blockIdx.x;
#pragma unroll
    for (int u = 0; u < PF; u++)
        if (u * THREADS < total_units) early[u] = load_unit(block_of(g), tid + u * THREADS);
    if constexpr (AT_ONCE) {
#pragma unroll
        for (int u = 0; u < WF; u++)
            if (u * THREADS < halves / 8) first[u] = load_weights(tid + u * THREADS);
    }

    // ---- weights: into LDS, then packed in the order the MFMAs take them --------------------------------------------------
    _Float16* raw = (_Float16*)(smem + p.raw_offset);
    if constexpr (AT_ONCE) {
#pragma unroll
        for (int u = 0; u < WF; u++)
            if (tid + u * THREADS < halves / 8) ((uintx4*)raw)[tid + u * THREADS] = first[u];
    }
    for (int i = tid + WF * THREADS; i < halves / 8; i += THREADS) ((uintx4*)raw)[i] = ((const uintx4*)src)[i];
    for (int i = (halves & ~7) + tid; i < halves; i += THREADS) raw[i] = src[i];
    __syncthreads();
    {
        // one step of one MFMA tile at a time, a lane's pair of pixels in four dwords read around it and shifted into place
        // (half by half the 7x7 layer spent 2 us here); what lies beyond the pair is read (LDS that the plan reserves) and
        // masked
        auto pack = [&](int s, int j) {
            const int chunk = 4 * s + q, kh = p.by_pairs.div(chunk), kw = 2 * (chunk - kh * p.pairs);
            const int n = channel_of(j, r);
            const bool ok = n < ocs && chunk < p.chunks;
            const int at = ok ? n * filter + (kh * p.kW + kw) * p.IC : 0, odd = (at & 1) * 2;
            const unsigned* from = (const unsigned*)raw + (at >> 1);
            const unsigned w0 = from[0], w1 = from[1], w2 = from[2], w3 = from[3];
            const unsigned h0 = __builtin_amdgcn_alignbyte(w1, w0, odd), h1 = __builtin_amdgcn_alignbyte(w2, w1, odd);
            const unsigned h2 = __builtin_amdgcn_alignbyte(w3, w2, odd), h3 = w3;      // (four channels: never odd)
            uintx4 v;
            if (p.IC == 3) v = uintx4{h0, h1 & 0xffffu, h1 >> 16 | h2 << 16, h2 >> 16};
            else if (p.IC == 4) v = uintx4{h0, h1, h2, h3};
            else if (p.IC == 2) v = uintx4{h0, 0, h1, 0};
            else v = uintx4{h0 & 0xffffu, 0, h0 >> 16, 0};
            const unsigned one = ok ? 0xffffffffu : 0u, two = ok && kw + 1 < p.kW ? 0xffffffffu : 0u;
            v[0] &= one, v[1] &= one, v[2] &= two, v[3] &= two;
            *(uintx4*)(smem + p.packed_offset + s * STEP_BYTES + (j * 64 + lane) * 16) = v;
        };
        const int items = p.steps * NT;
#pragma unroll 2
        for (int i = wave; i < items; i += WAVES) pack(i / NT, i % NT);
    }
    __syncthreads();
    constexpr int KR = KS > 0 ? KS : 1;
    half8 bw[KR][NT];
    if constexpr (KS > 0) {
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
                bw[s][j] = half8{0, 0, 0, 0, 0, 0, 0, 0};
                if (s < p.steps) bw[s][j] = *(const half8*)(smem + p.packed_offset + s * STEP_BYTES + (j * 64 + lane) * 16);
            }
        __syncthreads();                                       // the patch takes the weights' place
    }
    if (tid == 0) *(uintx4*)smem = uintx4{0, 0, 0, 0};

    const bool wide = p.OC % 8 == 0;                           // y is 16-byte aligned then (checked on the host)
    // byte offset of this lane's chunk of step s from a pixel's corner (negative: no such chunk), and the mask of the
    // pair's second pixel
    auto chunk_offset = [&](int s) -> int {
        const int chunk = 4 * s + q;
        const int kh = p.by_pairs.div(chunk), kp = chunk - kh * p.pairs;
        return chunk < p.chunks ? (kh * p.patch_cols + 2 * kp) * 8 : -1;
    };
    auto second_mask = [&](int s) -> unsigned {
        const int chunk = 4 * s + q;
        const int kp = chunk - p.by_pairs.div(chunk) * p.pairs;
        return 2 * kp + 1 < p.kW ? 0xffffffffu : 0u;
    };
    int pixels = 0, width = 1;                                 // of the current block
    _Float16* out = p.y;
    auto pixel_of = [&](int m) -> int2 {                       // block row and column of a pixel of the block
        const int oh = width == p.cols ? p.by_cols.div(m) : m / width;
        return int2{oh, m - oh * width};
    };
    auto corner = [&](int tile) -> int {                       // LDS offset of the lane's pixel of a tile
        const int m = tile * 16 + r;
        const int2 at = pixel_of(m < pixels ? m : pixels - 1);
        return ZERO_BYTES + (at.x * p.stride * p.patch_cols + at.y * p.stride) * 8;
    };
    auto fragment = [&](int at, int off, unsigned mask) -> half8 {
        uintx4 v = read16(smem + (off < 0 ? 0 : at + off));
        v[2] &= mask;
        v[3] &= mask;
        return __builtin_bit_cast(half8, v);
    };
    auto store = [&](int tile, const floatx4 (&acc)[NT]) {
        const int m = tile * 16 + r;
        if (m >= pixels) return;
        size_t px = m;
        if (p.col_blocks > 1) {
            const int2 at = pixel_of(m);
            px = (size_t)at.x * p.OW + at.y;
        }
#pragma unroll
        for (int i = 0; i < NT / 2; i++) {
            const floatx4 lo = acc[2 * i], hi = acc[2 * i + 1];
            const half8 h = {(_Float16)lo[0], (_Float16)lo[1], (_Float16)lo[2], (_Float16)lo[3],
                             (_Float16)hi[0], (_Float16)hi[1], (_Float16)hi[2], (_Float16)hi[3]};
            const int n = i * 32 + q * 8;
            _Float16* dst = out + px * p.OC + n;
            if (wide && n + 8 <= ocs) {
                *(uintx4*)dst = __builtin_bit_cast(uintx4, h);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (n + e < ocs) dst[e] = h[e];
            }
        }
    };

    constexpr int OFFS = KS > 0 ? KS : 1;
    int off[OFFS];
    unsigned second = 0;                                       // bit s: the pair of step s has its second pixel
#pragma unroll
    for (int s = 0; s < OFFS; s++) {
        off[s] = chunk_offset(s);
        second |= second_mask(s) & (1u << s);
    }
    auto mask_of = [&](int s) -> unsigned { return (unsigned)((int)(second << (31 - s)) >> 31); };

    while (true) {
        const Block now = block_of(g);
        int t = tid;                                           // keeps what follows from it out of registers across the loop
        asm volatile("" : "+v"(t));
#pragma unroll
        for (int u = 0; u < PF; u++)
            if (u * THREADS < total_units) store_unit(now, t + u * THREADS, early[u]);
#pragma unroll 1
        for (int i = t + PF * THREADS; i < total_units; i += THREADS) store_unit(now, i, load_unit(now, i));
        __syncthreads();
        g += gridDim.x;
        const bool more = g < p.blocks;
        if (more) {
#pragma unroll
            for (int u = 0; u < PF; u++)
                if (u * THREADS < total_units) early[u] = load_unit(block_of(g), t + u * THREADS);
        }
        const int rows = (p.OH - now.oh0) < p.rows ? (p.OH - now.oh0) : p.rows;
        width = (p.OW - now.ow0) < p.cols ? (p.OW - now.ow0) : p.cols;
        pixels = rows * width;
        const int tiles = (pixels + 15) / 16;
        out = p.y + (((size_t)now.image * p.OH + now.oh0) * p.OW + now.ow0) * p.OC + oc0;

        if constexpr (KS > 0) {
            half8 a[KR];
            if (wave < tiles) {
                const int at = corner(wave);
#pragma unroll
                for (int s = 0; s < KS; s++) a[s] = fragment(at, off[s], mask_of(s));
            }
            for (int tile = wave; tile < tiles; tile += WAVES) {
                floatx4 acc[NT];
#pragma unroll
                for (int j = 0; j < NT; j++) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
                const int at = corner(tile + WAVES);           // past the last tile: the last pixel again, not used
#pragma unroll
                for (int s = 0; s < KS; s++) {
#pragma unroll
                    for (int j = 0; j < NT; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bw[s][j], a[s], acc[j], 0, 0, 0);
                    a[s] = fragment(at, off[s], mask_of(s));   // the next tile's, into the registers just used
                }
                store(tile, acc);
            }
        } else {
            constexpr int MT = 4;                              // tiles in flight: a fragment of weights serves four of pixels
            for (int tile = wave * MT; tile < tiles; tile += WAVES * MT) {
                floatx4 acc[MT][NT];
                int at[MT];
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    at[i] = corner(tile + i);
#pragma unroll
                    for (int j = 0; j < NT; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
                }
                half8 a[2][MT], b[2][NT];
                auto read_step = [&](int s, half8 (&av)[MT], half8 (&bv)[NT]) {
                    const int o = chunk_offset(s);
                    const unsigned mask = second_mask(s);
#pragma unroll
                    for (int i = 0; i < MT; i++) av[i] = fragment(at[i], o, mask);
#pragma unroll
                    for (int j = 0; j < NT; j++)
                        bv[j] = *(const half8*)(smem + p.packed_offset + s * STEP_BYTES + (j * 64 + lane) * 16);
                };
                auto multiply = [&](const half8 (&av)[MT], const half8 (&bv)[NT]) {
#pragma unroll
                    for (int j = 0; j < NT; j++)
#pragma unroll
                        for (int i = 0; i < MT; i++)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bv[j], av[i], acc[i][j], 0, 0, 0);
                };
                read_step(0, a[0], b[0]);
                for (int s = 0; s < p.steps; s += 2) {         // a step is read while the one before it is multiplied
                    read_step(s + 1 < p.steps ? s + 1 : s, a[1], b[1]);
                    multiply(a[0], b[0]);
                    if (s + 1 < p.steps) {
                        read_step(s + 2 < p.steps ? s + 2 : s, a[0], b[0]);
                        multiply(a[1], b[1]);
                    }
                }
#pragma unroll
                for (int i = 0; i < MT; i++)
                    if (tile + i < tiles) store(tile + i, acc[i]);
            }
        }
        if (!more) break;
        __syncthreads();                                       // every wave is done with the patch
    }
}

// ---- host side ------------------------------------------------------------------------------------------------------
struct Plan {
    Params p;
    int ks;            // kernel variant: 2, 4 or 7 steps of weights in registers, 0: weights in LDS
    int nt;            // and MFMA tiles of channels per workgroup
    int lds_bytes;
    int grid;          // workgroups per block of output channels
};

inline size_t align16(size_t n) { return (n + 15) & ~(size_t)15; }

// Whether this kernel is the faster path for a layer that it can run.  It stages the input again for every 64 output channels:
// in units of four pixels for three channels, pixel by pixel for the others, which is what those are bound by once each output
// pixel has `staged` input pixels moved for it over all channel blocks.  us per launch, the fastest of fifteen configurations of
// the general path / this kernel, 64 images of 112 x 112, stride 4:
//   3 -> 1024 channels        3x3  43 / 28, 11x11 123 / 104
//   4 -> 256 | 512 (staged 56 | 112)    1x1  18 / 17 | 24 / 29, 7x7 33 / 29 | 50 / 55
//   1 -> 128 | 256 (staged 28 - 37 | 56 - 70)   3x3  12 / 10 | 15 / 14, 7x7 16 / 15 | 19 / 23
//   1 -> 64 | 256, 11x11 (17 steps)   23 / 16 | 29 / 39; 8 images of 224 x 224, stride 2, 13x13 -> 128 | 256  47 / 32 | 54 / 60
// Filters of more than seven steps have their weights in LDS and a longer way to the first result: of one channel, 64 x 64 at
// batch 1 | 2 | 4 | 8, 9x9 8.4 / 8.6 | 8.5 / 8.7 | 11 / 10 | 13 / 10, 11x11 8.7 / 10.5 | 9.0 / 10.5 | 11 / 11 | 18 / 12, of two
// the same at half as many pixels.
// Results beyond the 256 MB memory-side cache in rows of more than 512 channels: the 128-byte pieces of a pixel that a
// workgroup writes reach HBM at 3.9 - 5.0 TB/s, the general path's 512-byte ones faster than it loses by its copies where
// the filter is 1x1 (4 x 256 x 256 x 3 -> 2048 216 / 277, -> 4096 391 / 516), about level for 3x3 ones from 2048 channels on.
inline bool is_faster(long long pixels, double staged, int IC, int OC, int steps) {
    if (OC > 512 && pixels * OC * 2 > (256LL << 20) && !(IC == 3 && steps >= (OC <= 1024 ? 2 : 4))) return false;
    if (IC == 3) return true;
    if (IC == 4) return staged <= 96.0;
    if (steps <= 7) return staged <= 48.0;
    return staged <= 24.0 && pixels * IC >= 16384 && (steps <= 17 || OC <= 2 * OC_BLOCK);
}

// The split of a layer over workgroups; false where the layer does not fit this kernel (more than four channels, filters or
// rows beyond what LDS holds) or another path is the faster one.
inline bool make_plan(Plan& plan, int batch, int H, int W, int IC, int OC, int kH, int kW, int stride, int pad) {
    if (IC > 4 || (long long)batch * H * W * IC * 2 >= 0x7ffffff0LL) return false;
    const int OH = (H + 2 * pad - kH) / stride + 1, OW = (W + 2 * pad - kW) / stride + 1;
    const long long pairs = (kW + 1) / 2, chunks = kH * pairs, steps = (chunks + 3) / 4;
    if (steps > MAX_STEPS || (long long)batch * OH * OW > 0x7fffffffLL) return false;
    const int ks = steps <= 2 ? 2 : steps <= 4 ? 4 : steps <= 7 ? 7 : 0, waves = threads_of(ks) / 64, per_wave = ks ? 1 : 4;
    const int oc_blocks = (OC + OC_BLOCK - 1) / OC_BLOCK;
    if (oc_blocks > 65535) return false;
    // input pixels under the output, borders included, per output pixel and channel block
    const double staged = ((double)(OH - 1) * stride + kH) * ((double)(OW - 1) * stride + kW) / ((double)OH * OW) * oc_blocks;
    if (!is_faster((long long)batch * OH * OW, staged, IC, OC, (int)steps)) return false;
    // 96 channels per workgroup where one then holds all of a pixel and there are many: written by two, its 64 and 32 channels
    // are not whole 128-byte lines, and the input is staged twice.  us per launch at 64 / 96, three channels -> 96: 4 x 224 x 224
    // 3x3 16.2 / 11.2, 32 x 224 x 224 5x5 stride 2 25.7 / 21.2; 77k pixels 8.4 / 8.3, 900 - 23k pixels 5.0 / 5.8, 5.8 / 6.3; with
    // seven steps (one workgroup per CU, for the registers) 28.5 / 28.2 at 307k pixels, 9.9 / 10.7 at 30k.  One, two and four channels
    // have not been measured at 96 and stay at 64
    const int nt = IC == 3 && ks > 0 && ks <= 4 && OC > 64 && OC <= 96 && (long long)batch * OH * OW >= (1 << 17) ? 6 : 4;
    const int nt_blocks = (OC + 16 * nt - 1) / (16 * nt);
    const size_t raw = align16((size_t)16 * nt * kH * kW * IC * 2), packed = (size_t)steps * step_bytes(nt);
    double best = 0.0;
    Params& p = plan.p;
    // candidates: this runs on every call, so a few of them (a search over all rows took longer than the small layers).
    // Whole rows measure fastest wherever there are enough of them; rows are cut into halves, quarters ... only for
    // layers of few rows (batch 1)
    static const int row_counts[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32, 40, 48};
    const int max_halve = (long long)batch * OH * oc_blocks < 512 ? 3 : 0;
    for (int halve = 0; halve <= max_halve; halve++) {
        const int cols = halve == 0 ? OW : ((OW >> halve) + 15) / 16 * 16;
        if (halve && (cols >= OW || cols < 16)) break;
        const int col_blocks = (OW + cols - 1) / cols;
        const long long patch_cols = ((long long)(cols - 1) * stride + 2 * pairs + 1) / 2 * 2;
        for (const int rows : row_counts) {
            if (rows > OH) break;
            const long long patch = ZERO_BYTES + ((long long)(rows - 1) * stride + kH) * patch_cols * 8;
            // weights in registers: raw and packed weights lie where the patch goes later; in LDS: packed weights behind
            // the patch, the raw ones in its place
            const long long lds = ks ? (patch > (long long)(raw + packed) ? patch : (long long)(raw + packed))
                                     : (long long)align16((size_t)(patch > (long long)raw ? patch : (long long)raw)) + (long long)packed;
            if (lds > LDS_MAX) break;
            int resident = (int)(LDS_MAX / lds);
            if (resident > resident_of(ks, nt)) resident = resident_of(ks, nt);
            const long long blocks = (long long)batch * ((OH + rows - 1) / rows) * col_blocks;
            if (blocks > 0x7fffffffLL) continue;
            const long long slots = 256LL * resident, wgs = blocks * nt_blocks;
            const long long rounds = (wgs + slots - 1) / slots, grid = (blocks + rounds - 1) / rounds;
            // cycles: the weights once per workgroup, then per block its patch and its MFMAs, which the workgroups of a
            // compute unit share
            const long long sharing = (grid * nt_blocks + 255) / 256;
            const double per_block = (double)patch / 20.0 + 500.0;
            const long long tile_rounds = (((long long)rows * cols + 15) / 16 + waves * per_wave - 1) / (waves * per_wave) * per_wave;
            const double multiply = (double)tile_rounds * (waves / 4) * (double)steps * nt * 22.0;
            const double t = 300.0 * (double)steps + (double)rounds * (per_block + (double)sharing * multiply);
            if (best == 0.0 || t < best) {
                best = t;
                p.rows = rows;
                p.cols = cols;
                p.row_blocks = (OH + rows - 1) / rows;
                p.col_blocks = col_blocks;
                p.blocks = (int)blocks;
                p.patch_rows = (rows - 1) * stride + kH;
                p.patch_cols = (int)patch_cols;
                plan.lds_bytes = (int)lds;
                plan.grid = (int)grid;
            }
        }
    }
    if (best == 0.0) return false;
    p.H = H; p.W = W; p.IC = IC; p.OC = OC; p.OH = OH; p.OW = OW; p.kH = kH; p.kW = kW; p.stride = stride; p.pad = pad;
    p.pairs = (int)pairs; p.chunks = (int)chunks; p.steps = (int)steps;
    p.raw_offset = 0;
    p.packed_offset = ks ? (int)raw : plan.lds_bytes - (int)packed;
    p.unit_pixels = IC == 3 && (long long)batch * H * W >= 8 ? 4 : 1;
    p.x_bytes = (unsigned)((long long)batch * H * W * IC * 2);
    // a row's units start up to unit_pixels - 1 pixels in front of the patch
    const int units = (p.patch_cols + p.unit_pixels - 1 + p.unit_pixels - 1) / p.unit_pixels;
    p.by_cols = helix_fastdiv::make(p.cols);
    p.by_row_blocks = helix_fastdiv::make(p.row_blocks);
    p.by_col_blocks = helix_fastdiv::make(p.col_blocks);
    p.by_pairs = helix_fastdiv::make((int)pairs);
    p.by_units = helix_fastdiv::make(units);
    plan.ks = ks;
    plan.nt = nt;
    return true;
}

template <int KS, int NT>
inline int launch_steps(const Plan& plan, hipStream_t s) {
    static int rc = (int)hipFuncSetAttribute((const void*)helix_conv_thin_f16_kernel<KS, NT>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX);
    if (rc) return rc;
    const dim3 grid((unsigned)plan.grid, (unsigned)((plan.p.OC + 16 * NT - 1) / (16 * NT)), 1);
    hipLaunchKernelGGL((helix_conv_thin_f16_kernel<KS, NT>), grid, dim3(threads_of(KS)), plan.lds_bytes, s, plan.p);
    return (int)hipGetLastError();
}

// x, w: 16-byte aligned; y: 16-byte aligned where OC is a multiple of 8.
inline int launch(Plan& plan, const void* x, const void* w, void* y, hipStream_t s) {
    plan.p.x = (const _Float16*)x;
    plan.p.w = (const _Float16*)w;
    plan.p.y = (_Float16*)y;
    switch (plan.ks * 8 + plan.nt) {
        case 2 * 8 + 4: return launch_steps<2, 4>(plan, s);
        case 2 * 8 + 6: return launch_steps<2, 6>(plan, s);
        case 4 * 8 + 4: return launch_steps<4, 4>(plan, s);
        case 4 * 8 + 6: return launch_steps<4, 6>(plan, s);
        case 7 * 8 + 4: return launch_steps<7, 4>(plan, s);
        default: return launch_steps<0, 4>(plan, s);
    }
}

}  // namespace
}  // namespace helix_conv_thin
