// Tiles of an image and their hand-out to the one-wave blocks of the megakernel
// and the adjoint.
#ifndef NOOR_TILE_FEED_H
#define NOOR_TILE_FEED_H

#include <stdint.h>

#ifdef __HIPCC__
#define NOOR_HD __host__ __device__ __forceinline__
#else
#define NOOR_HD inline
#endif

namespace noor {

// The launch has at most as many blocks as the GPU holds at once; a block that
// is done with its tile takes another one (with the tiles dealt out in advance
// the 1080p terrain frame takes 3.6 instead of 3.0 ms).  The tiles are split
// over kTileGroups groups with a counter each, block b taking from group
// b % kTileGroups, one group per XCD: returning atomics on one address are
// 11.7 ns apart, which with one counter made a frame whose rays all miss take
// 0.40 ms at 1920x1080 and 1.51 at 3840x2160 (0.19 and 0.45 with 8 groups, 0.15
// and 0.39 with 16, 0.10 and 0.29 with the tiles dealt out; 16 take 8.4 instead
// of 8.2 ms for the terrain at 3840x2160, one 8.4).  A group owns one tile of
// every kTileGroups, another one in each run of them, so that no group gets the
// same columns of every row; a block whose group has run out takes from the
// others.
constexpr uint32_t kTileGroups = 8;

// Tile of entry i of group g, and the entries of a group.
NOOR_HD uint32_t group_tile(uint32_t g, uint32_t i) { return i * kTileGroups + ((g + i) & (kTileGroups - 1)); }
NOOR_HD uint32_t group_size(uint32_t g, uint32_t tiles) {
    const uint32_t n = tiles / kTileGroups;
    return n + (((g + n) & (kTileGroups - 1)) < tiles % kTileGroups ? 1u : 0u);
}

// How many blocks cover `tiles` tiles: one each, or what `waves` resident waves
// allow, the same number for every group.
NOOR_HD uint32_t tile_blocks(uint32_t tiles, uint32_t waves) {
    if (tiles <= waves) return tiles;
    return waves < kTileGroups ? kTileGroups : waves / kTileGroups * kTileGroups;
}

// Entries handed out of each group beyond the blocks' first, blocks of each
// group that have ended, and groups that have: the last block clears all, so a
// launch needs no memset before it.  Each on a 256-byte line of its own.
struct TileWork {
    struct Line {
        uint32_t v, pad[63];
    };
    Line next[kTileGroups], done[kTileGroups], groups;
};

#ifdef __HIPCC__
// A one-wave block's first tile.
__device__ __forceinline__ uint32_t first_tile(uint32_t tiles) {
    if (gridDim.x >= tiles) return blockIdx.x;
    return group_tile(blockIdx.x % kTileGroups, blockIdx.x / kTileGroups);
}
// Its next one; `tiles` when there is none.  Called by all lanes of the wave.
__device__ __forceinline__ uint32_t next_tile(TileWork* work, uint32_t tiles) {
    if (gridDim.x >= tiles) return tiles;  // every tile was some block's first
    const uint32_t lane = threadIdx.x & 63u, dealt = gridDim.x / kTileGroups;  // (blocks of each group)
    uint32_t g = blockIdx.x % kTileGroups;
    // groups that may have tiles left: each turn takes a tile or one of them away
    for (uint32_t left = (1u << kTileGroups) - 1u; left != 0u;) {
        uint32_t n = 0;
        if (lane == 0) n = atomicAdd(&work->next[g].v, 1u);
        const uint32_t i = dealt + (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
        if (i < group_size(g, tiles)) return group_tile(g, i);
        // this group has run out: look at all of them, take the next one that has not
        left &= ~(1u << g);
        bool some = false;
        if (lane < kTileGroups)
            some = dealt + __hip_atomic_load(&work->next[lane].v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
                   group_size(lane, tiles);
        left &= (uint32_t)__ballot(some);
        const uint32_t after = left & ~((2u << g) - 1u);
        g = (uint32_t)__builtin_ctz((after ? after : left) | (1u << kTileGroups));
    }
    return tiles;
}
// Every block calls it once, after its last next_tile().
__device__ __forceinline__ void tiles_done(TileWork* work, uint32_t tiles) {
    if (gridDim.x >= tiles || (threadIdx.x & 63u) != 0) return;
    const uint32_t g = blockIdx.x % kTileGroups;
    if (atomicAdd(&work->done[g].v, 1u) != gridDim.x / kTileGroups - 1u) return;
    atomicExch(&work->done[g].v, 0u);
    if (atomicAdd(&work->groups.v, 1u) != kTileGroups - 1u) return;
    for (uint32_t k = 0; k < kTileGroups; ++k) atomicExch(&work->next[k].v, 0u);
    atomicExch(&work->groups.v, 0u);
}
#endif

}  // namespace noor
#endif
