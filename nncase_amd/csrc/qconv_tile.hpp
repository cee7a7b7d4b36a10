// The window kernel that keeps a tile's input in LDS (qconv_tile.hip): what a launch of it is planned as.
#pragma once

#include "qconv_wide.hpp"

namespace nnhip {

__device__ __forceinline__ int tile_div(int p, uint32_t mul) { return (int)(__umul24((uint32_t)p, mul) >> 20); } // make_tile_div

// LDS for the sums of `units` results of each wave that the groups of a split reduction pass on.
constexpr int tile_part_bytes(int units, int waves, int groups) { return units * (groups - 1) * waves * 1024; }

struct TileArgs {
    int th, tw;                    // output tile
    int hr, hc;                    // input rows / columns under it
    int half;                      // input columns per column phase (stride 2: column c lies at (c & 1) * half + c / 2, so that
                                   // neighbouring output pixels read neighbouring LDS pixels)
    int pitch, row_pitch;          // bytes of an LDS pixel (an odd number of 16-byte pieces: eight lanes, eight banks) / row
    int pieces;                    // 16-byte pieces per pixel
    int apart, dc, dr;             // whole pixels that a block's threads cover at once, and that as a step in (column, row)
    int row_bytes;                 // of the tensor
    int tile_off;
    uint32_t d_pieces, d_hc, d_tw; // of make_tile_div
    FastDiv d_tx, d_txy, d_nchunks, d_rest;
};

// Pixels x channels of a block; by n: its k-steps shared by n groups of waves.
enum TileShape {
    kTile128x32, kTile64x32, kTile32x64, kTile128x128, kTile64x128,
    kTile32x32by2, kTile32x32by4, kTile16x32by4, kTile32x64by2, kTile32x64by4, kTile16x64by4,
    kTileNone
};

struct TilePlan {
    TileShape shape = kTileNone;
    TileArgs t;
    int tiles; // of the whole batch
    size_t lds;
};

// The plan of a call (the same for every group of a grouped layer); shape kTileNone: not a layer of this kernel.
TilePlan plan_qconv_tile(const nncase_hip_ctx *ctx, const IgemmArgs &a, int tiles, int nchunks);
int launch_qconv_tile(nncase_hip_ctx *ctx, const IgemmArgs &a, const TilePlan &plan, int nchunks);

} // namespace nnhip
