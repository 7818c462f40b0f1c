// What the ring templates of both backends share (MI355X_FP16/gemm_ring.hip, MI355X_FP32/gemm_ring.hip): copies from global memory
// into LDS that pass no register, their waits, and the walk of a launch's tiles.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace helix_ring {

typedef int intx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) unsigned char* lds_ptr_t;

constexpr int GROUP_ROWS = 4, NUM_XCD = 8;
constexpr int OOB_OFFSET = 0x7ffffff0;              // byte offset, of a whole copy, beyond any buffer (less than 2 GiB each): zeros

// 128-bit buffer descriptor as four dwords: base address (48 bits), stride 0, byte count, raw-buffer flags
__device__ __forceinline__ intx4 raw_rsrc(const void* base, unsigned bytes) {
    const unsigned long long a = (unsigned long long)base;
    return intx4{(int)(unsigned)a, (int)((a >> 32) & 0xffffu), (int)bytes, 0x00020000};
}

// One 16-byte-per-lane copy into LDS: lane l's data lands at LDS byte lds_addr + 16 l (wave-uniform, through M0), zeros where its
// offset is beyond the buffer.  From inline assembly, so that the compiler neither orders LDS reads behind it nor counts it in
// its own waits: completion is waited for by hand, in front of the barrier that publishes it.
__device__ __forceinline__ void copy16(intx4 rsrc, unsigned lds_addr, int offset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(offset), "s"(rsrc)
                 : "memory", "m0");
}

// s_waitcnt vmcnt(COPIES_LEFT), and lgkmcnt(0) where LDS_TOO
template <int COPIES_LEFT, bool LDS_TOO>
__device__ __forceinline__ void wait() {
    __builtin_amdgcn_s_waitcnt((COPIES_LEFT & 15) | (7 << 4) | ((LDS_TOO ? 0 : 15) << 8) | ((COPIES_LEFT >> 4) << 14));
}

// The barrier in the middle of a tile: what this wave read and what it copied for the next tile is complete on either side of it
template <int COPIES_LEFT>
__device__ __forceinline__ void wait_and_meet() {
    wait<COPIES_LEFT, true>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// Workgroup ids are dealt round-robin to the 8 XCDs: each is given a compact run of tiles, walked in column-major groups of rows.
// False for the ids beyond the last tile.
__device__ __forceinline__ bool tile_of(int id, int tiles_m, int tiles_n, int* tm, int* tn) {
    const int ntiles = tiles_m * tiles_n, per_xcd = (ntiles + NUM_XCD - 1) / NUM_XCD;
    const int slot = id / NUM_XCD, pid = id % NUM_XCD * per_xcd + slot;
    if (slot >= per_xcd || pid >= ntiles) return false;
    const int group_tiles = GROUP_ROWS * tiles_n, first_m = pid / group_tiles * GROUP_ROWS, in_group = pid % group_tiles;
    const int rows = (tiles_m - first_m) < GROUP_ROWS ? (tiles_m - first_m) : GROUP_ROWS;
    *tm = first_m + in_group % rows;
    *tn = in_group / rows;
    return true;
}

}  // namespace helix_ring
