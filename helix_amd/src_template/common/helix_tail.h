// The last round of a tile launch, partitioned along K (the FP32 tile template).
//
// A launch of T output tiles keeps the 256 compute units busy for ceil(T / 256) rounds; T just above a multiple of 256
// leaves most of them idle through the last one (25088 x 128 FP32 in 64 x 64 tiles: 784 tiles, 16 of them in a fourth
// round).  Partitioning every tile along K makes the rounds finer but writes the whole result to the workspace several
// times over.  Here only the R = T mod 256 tiles beyond the whole rounds are partitioned:
//   * the workgroups behind the whole tiles are their pieces, `splits` per tile, each one K range of one tile, which go to
//     the workspace as FP32 partial tiles ([tile][split][row][column]).  (Pieces in front of the whole tiles measured the
//     same on 18 of 28 launches, 3 - 6 % slower on 8 and 5 - 6 % faster on 2);
//   * a second kernel, one workgroup per 1024 elements, adds the partials in partition order (deterministic) and stores
//     the result.  A second kernel rather than the in-launch sum of helix_splitk.h: the partials are few, so all compute
//     units add them in 1 - 2 us, and there is no counter that launches on several streams would share.
// The workspace is optional: without it the launch runs unpartitioned.
//
// Built into the FP16 template as well and taken out again: it took a third off launches just above a round (661 x 11008 x
// 4096 in 256 x 128 tiles: 258 tiles, 98 -> 69 us), but there a tile of another size that needs less than one round was
// faster on each of eight problems (256 x 192: 174 tiles, 65 us), and the larger kernels spilled.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace helix_tail {

constexpr int COMPUTE_UNITS = 256, MAX_SPLITS = 8;

typedef float floatx4 __attribute__((ext_vector_type(4)));

struct Plan {
    int tiles;    // R: tiles that are partitioned (the last R tile numbers); 0: none
    int splits;   // pieces per tile
    int k_per;    // K extent of a piece
    int ids;      // workgroup ids given to pieces, a multiple of 8 (some of them idle)
};

// Workgroup id -> tile number and piece.  Ids are dealt round-robin to the 8 XCDs; each XCD is given a compact run of the
// whole tiles (their number is a multiple of 256), and the pieces of a tile, which read the same panels, share an XCD.
struct Unit {
    int tile, tail_tile, split;   // split < 0: a whole tile; tail_tile: number of the tile among the partitioned ones
    bool idle;
};

__device__ __forceinline__ Unit unit_of_workgroup(const Plan& t, int ntiles) {
    const int id = (int)blockIdx.x, whole = ntiles - t.tiles;
    if (id < whole) return Unit{(id % 8) * (whole / 8) + id / 8, 0, -1, false};
    const int xcd = id % 8, j = (id - whole) / 8, slot = j / t.splits;
    const int per = t.tiles / 8, rem = t.tiles % 8;
    const int n = xcd * per + (xcd < rem ? xcd : rem) + slot;
    return Unit{whole + n, n, j - slot * t.splits, slot >= per + (xcd < rem ? 1 : 0)};
}

// Tile number -> tile row and column: column-major within groups of GROUP tile rows, so that the tiles in flight on an
// XCD share A and B panels in its L2.
template <int GROUP>
__device__ __forceinline__ int2 tile_position(int pid, int tiles_m, int tiles_n) {
    const int group_tiles = GROUP * tiles_n;
    const int first_m = (pid / group_tiles) * GROUP;
    const int gsize = (tiles_m - first_m) < GROUP ? (tiles_m - first_m) : GROUP;
    const int in_group = pid % group_tiles;
    return int2{first_m + in_group % gsize, in_group / gsize};
}

namespace {   // internal linkage: every library carries its own copy

// Adds the pieces of the partitioned tiles: thread = four consecutive columns of one tile row.
template <int TILE_ROWS, int TILE_COLS, int GROUP>
__global__ __launch_bounds__(256) void helix_tail_reduce_kernel(const float* ws, float* C, int M, int N, int ldc, int tiles_m,
                                                                int tiles_n, int first_tile, int splits) {
    constexpr int CHUNKS = TILE_ROWS * TILE_COLS / 4, PER_ROW = TILE_COLS / 4;
    const int c = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (c >= CHUNKS) return;
    const int2 at = tile_position<GROUP>(first_tile + (int)blockIdx.y, tiles_m, tiles_n);
    const int row = at.x * TILE_ROWS + c / PER_ROW, col = at.y * TILE_COLS + (c % PER_ROW) * 4;
    if (row >= M || col >= N) return;
    const floatx4* part = (const floatx4*)ws + (size_t)blockIdx.y * splits * CHUNKS + c;
    floatx4 v[MAX_SPLITS];
#pragma unroll
    for (int k = 0; k < MAX_SPLITS; k++)          // all loads in flight before the first addition
        if (k < splits) v[k] = __builtin_nontemporal_load(part + (size_t)k * CHUNKS);
    floatx4 sum = v[0];
#pragma unroll
    for (int k = 1; k < MAX_SPLITS; k++)
        if (k < splits) {
            sum[0] += v[k][0]; sum[1] += v[k][1]; sum[2] += v[k][2]; sum[3] += v[k][3];
        }
    float* dst = C + (size_t)row * ldc + col;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (col + e < N) dst[e] = sum[e];
}

}  // namespace

// ---- host side --------------------------------------------------------------------------------------------------
// What a template knows about its launches: seconds a round of 256 workgroups takes per column of K and besides that, the
// shortest K range worth a workgroup, the second kernel's cost, and the bytes the partial tiles may take at most.
struct Model {
    double per_k, fixed, reduce_launch, reduce_bytes_per_s;
    int min_k;
    long long max_bytes;
};

// The pieces per tile that make a launch of `tiles` tiles of `elements` results shortest; 0 if the last round is not worth
// partitioning or would not be shorter than `unpartitioned` seconds by 1 - `gain` of them.  (The host scripts' cost models
// evaluate the same expression.)
inline int choose(const Model& m, long long tiles, int elements, int K, int block_k, double unpartitioned, double gain) {
    const long long rounds = tiles / COMPUTE_UNITS, rest = tiles % COMPUTE_UNITS;
    if (rounds < 1 || rest == 0) return 0;
    const int ktiles = (K + block_k - 1) / block_k;
    const double whole = (double)rounds * ((double)(ktiles * block_k) * m.per_k + m.fixed);
    int best = 0;
    double best_t = unpartitioned * gain;
    for (int s = 2; s <= MAX_SPLITS && K / s >= m.min_k; s++) {
        const int per = (ktiles + s - 1) / s;
        if ((ktiles + per - 1) / per != s) continue;          // the same pieces as a smaller s
        if (rest * s * elements * 4 > m.max_bytes) break;
        const double piece_rounds = (double)((rest * s + COMPUTE_UNITS - 1) / COMPUTE_UNITS);
        const double t = whole + piece_rounds * ((double)(per * block_k) * m.per_k + m.fixed) + m.reduce_launch +
                         (s + 1.0) * (double)rest * elements * 4.0 / m.reduce_bytes_per_s;
        if (t < best_t) {
            best_t = t;
            best = s;
        }
    }
    return best;
}

inline Plan make_plan(long long tiles, int K, int block_k, int splits) {
    Plan p{0, 0, 0, 0};
    if (splits < 2) return p;
    p.tiles = (int)(tiles % COMPUTE_UNITS);
    p.splits = splits;
    p.k_per = ((K + block_k - 1) / block_k + splits - 1) / splits * block_k;
    p.ids = 8 * ((p.tiles + 7) / 8) * splits;
    return p;
}

inline size_t workspace_bytes(long long tiles, int elements, int splits) {
    return splits < 2 ? 0 : (size_t)(tiles % COMPUTE_UNITS) * (size_t)splits * (size_t)elements * sizeof(float);
}

inline unsigned grid(const Plan& p, long long tiles) { return (unsigned)(tiles - p.tiles + p.ids); }

template <int TILE_ROWS, int TILE_COLS, int GROUP>
inline int reduce(const Plan& p, const float* ws, float* C, int M, int N, int ldc, int tiles_m, int tiles_n, hipStream_t s) {
    constexpr int CHUNKS = TILE_ROWS * TILE_COLS / 4;
    hipLaunchKernelGGL((helix_tail_reduce_kernel<TILE_ROWS, TILE_COLS, GROUP>), dim3((CHUNKS + 255) / 256, p.tiles),
                       dim3(256), 0, s, ws, C, M, N, ldc, tiles_m, tiles_n, tiles_m * tiles_n - p.tiles, p.splits);
    return (int)hipGetLastError();
}

}  // namespace helix_tail
