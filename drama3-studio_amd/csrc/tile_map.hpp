// Which tile of the moe_align map a workgroup of the tiled packed GEMMs takes.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace dmoe {

constexpr int kTileXcds = 8;  // workgroups go to the XCDs in turn

// Workgroups of a grid over `max_tiles` row tiles and `cols` column tiles.
inline unsigned tile_grid(int max_tiles, int cols) {
    return (unsigned)((max_tiles + kTileXcds - 1) / kTileXcds * kTileXcds) * (unsigned)cols;
}

struct TileWork {
    int e, m0, mc, ct;  // expert, first sorted pair, pairs, column tile
};

// An XCD takes a contiguous share of the row tiles, so the tiles of one expert
// read its weights through one L2, and walks them column tile by column tile,
// so a row tile's activations stay there too (tiles dealt to the XCDs in turn
// instead: a W4A16 layer at 600 tokens, E 32, H 4096, I 1536 390 us against 362).
// What the grid holds beyond the call's tiles comes last and exits (false)
// while the others finish.  Tiles lie in the order of their pairs, so the next
// one's start ends this one: no load waits for the expert's offsets.
__device__ __forceinline__ bool take_tile(const PackedGroupedArgs& a, int cols, TileWork& t) {
    const int count = *a.tile_count, valid = a.p.offsets[a.experts];
    const int x = (int)blockIdx.x % kTileXcds, j = (int)blockIdx.x / kTileXcds;
    const int lo = x * count / kTileXcds, n = (x + 1) * count / kTileXcds - lo;
    if (j >= n * cols) return false;
    t.ct = j / n;
    const int tile = lo + j - t.ct * n;
    t.e = a.tile_expert[tile];
    t.m0 = a.tile_m0[tile];
    const int next = a.tile_m0[min(tile + 1, count - 1)];
    t.mc = (tile + 1 < count ? next : valid) - t.m0;
    return true;
}

}  // namespace dmoe
