// Tiles of two elastic steps per launch (kernels_tile.hip): their shapes and
// the choice among them (host code).
#pragma once
#include <algorithm>
#include <vector>

namespace ds2d {

// A tile's halo columns and rows on each side, the rows it owns, and the cells
// of a window's frame that are never updated.
constexpr int TILE_HALO = 16, TILE_ROWS = 64 - 2 * TILE_HALO, TILE_KINDS = 4, TILE_FRAME = 4;

// Columns per wave and waves of the four tiles, and what one round of one
// workgroup per CU costs per launch of two steps (us, PML windows; measured
// on 251x101 windows, 1 to 26 of them; windows with the random boundary, whose
// launches take three quarters of that, are planned by the same costs).
struct TileKind {
    int k, nw;
    float us;
};
constexpr TileKind kTiles[TILE_KINDS] = {{3, 14, 9.2f}, {4, 12, 10.2f}, {4, 14, 12.1f}, {5, 12, 12.5f}};

struct TilePlan {
    int kind, cols;    // tile and its owned columns
    long long rounds;  // rounds of one workgroup per CU
    float us;          // estimate of one launch
};

// The tile whose rounds of the chip cost least for windows of nxp columns and nzp rows.
inline TilePlan plan_tiles(const std::vector<int>& nxp, int nzp, int ncu) {
    TilePlan best{0, 0, 0, 0.f};
    const long long zt = (std::max(nzp - 2 * TILE_FRAME, 0) + TILE_ROWS - 1) / TILE_ROWS;
    for (int v = 0; v < TILE_KINDS; ++v) {
        const int cols = kTiles[v].k * kTiles[v].nw - 2 * TILE_HALO;
        long long t = 0;
        for (int w : nxp) t += (std::max(w - 2 * TILE_FRAME, 0) + cols - 1) / cols * zt;
        const long long rounds = (t + ncu - 1) / ncu;
        const float us = rounds * kTiles[v].us;
        if (v == 0 || us < best.us) best = TilePlan{v, cols, rounds, us};
    }
    return best;
}

}  // namespace ds2d
