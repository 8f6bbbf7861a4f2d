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
// the 1080p terrain frame takes 3.5 instead of 2.85 ms).  The tiles are split
// over kTileGroups groups with a counter each, block b taking from group
// b % kTileGroups, one group per XCD: returning atomics on one address are
// 11.7 ns apart, which with one counter made a frame whose rays all miss take
// 0.40 ms at 1920x1080 and 1.51 at 3840x2160 (0.15 and 0.40 with eight; 0.10 and
// 0.29 with the tiles dealt out; sixteen made the terrain at 3840x2160 3%
// slower).  A group owns one tile of every kTileGroups, another one in each run
// of them, so that no group gets the same columns of every row; a block whose
// group has run out takes from the others.
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
// `dealt`: the blocks of each group, or 0 when every tile is some block's first
// and no counter is used (an argument of the launch: kept from the grid's size
// it cost the megakernel registers and 3% with the Wald test).
__device__ __forceinline__ uint32_t first_tile(uint32_t dealt) {
    if (dealt == 0u) return blockIdx.x;
    return group_tile(blockIdx.x % kTileGroups, blockIdx.x / kTileGroups);
}
// The block's next tile; `tiles` when there is none.  Called by all lanes of the
// wave.
__device__ __forceinline__ uint32_t next_tile(TileWork* work, uint32_t tiles, uint32_t dealt) {
    if (dealt == 0u) return tiles;
    uint32_t g = blockIdx.x % kTileGroups;
    for (uint32_t k = 0; k < kTileGroups; ++k, g = (g + 1) % kTileGroups) {
        const uint32_t size = group_size(g, tiles) - dealt;
        // (another group's counter is read first: most have run out as well by then)
        if (k != 0 && (uint32_t)__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(
                          &work->next[g].v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >= size)
            continue;
        uint32_t n = 0;
        if ((threadIdx.x & 63u) == 0) n = atomicAdd(&work->next[g].v, 1u);
        n = (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
        if (n < size) return group_tile(g, dealt + n);
    }
    return tiles;
}
// Every block calls it once, after its last next_tile().
__device__ __forceinline__ void tiles_done(TileWork* work, uint32_t dealt) {
    if (dealt == 0u || (threadIdx.x & 63u) != 0) return;
    const uint32_t g = blockIdx.x % kTileGroups;
    if (atomicAdd(&work->done[g].v, 1u) != dealt - 1u) return;
    atomicExch(&work->done[g].v, 0u);
    if (atomicAdd(&work->groups.v, 1u) != kTileGroups - 1u) return;
    for (uint32_t k = 0; k < kTileGroups; ++k) atomicExch(&work->next[k].v, 0u);
    atomicExch(&work->groups.v, 0u);
}
#endif

}  // namespace noor
#endif
