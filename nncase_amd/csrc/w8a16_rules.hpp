// Which kernel computes a W8A16 product, as plain host arithmetic that a test can hold against measured times without a device.
#pragma once

#include <algorithm>
#include <cstdint>

namespace nnhip {

constexpr int kRowsPieces = 4;                 // 512-element pieces of a token row in LDS: k <= 2048
constexpr int kRowsMaxK = kRowsPieces * 512;
constexpr int kTileMaxK = 5120;                // ten k-steps a wave
constexpr int rows_in_lds_pitch(int k) { return k * 2 + 16; } // bytes per token row: the padding spreads the rows over the banks

// A product of `rows` token rows (1 to 64) and a reduction of k (whole k-steps of 64); tiles: 16-channel tiles of the result (glu:
// SwiGLU, a gate and an up tile each).
struct W8Product {
    int rows, k, tiles;
    bool glu;
    int row_tiles() const { return (rows + 15) / 16; }
    int share() const { return (k / 64 + 7) / 8; } // k-steps of a wave where eight waves share a tile's reduction
};

// Whether the rows fit in LDS for the kernel that has a tile (pair) per wave (it is built for 16, 32 and 64 of them).
inline bool rows_fit_lds(const W8Product &p) {
    const int built = p.row_tiles() <= 2 ? p.row_tiles() : 4;
    return p.k <= kRowsMaxK && built * 16 * rows_in_lds_pitch(p.k) <= 128 * 1024;
}

// Whether a product over at most kRowsMaxK is computed with a tile's reduction split over a block's waves.  The sum's order depends
// on it, so it is asked for the rows' count and the matrix alone: the product, the one that normalises its rows and the one that rotates
// them agree bit for bit.  A block per tile and 16 rows repeats the rows' trip and its own set-up, a tile per wave leaves the device to
// few blocks; the line, in tiles per compute unit, is where the two took the same (us split / not, 256 units; k = 448 and below is one
// k-step a wave).  Plain: 4 rows, k = 448, 970 tiles 3.8 / 4.1; 13 of 192, 842 tiles 3.6 / 3.2; 14 of 640, 707 tiles 4.3 / 4.9; 26 of 384, 434
// tiles 4.2 / 4.0; 22 of 576, 509 tiles 4.9 / 5.5; 43 of 192, 285 tiles 3.7 / 4.6; 60 of 256, 493 tiles 5.7 / 5.1.  SwiGLU: 3 rows, k = 192, 940 pairs
// 4.6 / 4.5; 11 of 448, 890 pairs 5.2 / 5.9; 22 of 256, 529 pairs 5.8 / 5.4; 42 of 832, 552 pairs 9.3 / 10.6.
inline bool rows_take_split(const W8Product &p, int compute_units) {
    if (p.k > kRowsMaxK) return false;
    const int rt = p.row_tiles();
    const bool one_step = p.share() == 1;
    int quarters; // of a tile per compute unit
    if (!rows_fit_lds(p)) quarters = 20;
    else if (p.rows <= 8) quarters = p.glu || one_step ? 16 : 24;
    else if (rt == 1) quarters = p.glu ? 12 : one_step ? 10 : p.share() == 2 ? 12 : 16;
    else if (!one_step) quarters = 9;
    else quarters = rt == 2 ? 7 : p.glu ? 8 : 6;
    return 4 * p.tiles < quarters * compute_units;
}

// Whether a long reduction over few tiles is computed in tiles of 8 by 8 (and summed in their order, whichever kernel does it).
// They are four times the blocks of 16 by 16, each of which moves half as much: taken while all of them run at once, of nine and
// ten k-steps a wave.  us, 16 by 16 / 8 by 8, k = 4864, 896 columns: one row 5.3 / 4.4, 8 rows 6.2 / 5.7, 16 rows 7.9 / 5.6, 32 rows
// 7.9 / 8.4; shorter, 7 rows of 2240 to 1008 columns 3.7 / 4.6, 6 of 3776 to 1200 4.6 / 4.9.
inline bool sums_in_pairs(const W8Product &p, int compute_units) {
    return p.k > 4096 && p.k <= kTileMaxK && p.rows <= 16 && !p.glu && 2 * p.tiles * ((p.rows + 7) / 8) <= compute_units;
}

enum class W8Form {
    kTile,      // a tile (pair) per block, its reduction split over the waves, every request at once, the rows through LDS
    kTileLong,  // ... the rows read where they lie
    kSmallTile, // 8 channels by 8 rows per block
    kRowsInLds, // a tile (pair) per wave, rows in LDS
    kSplit,     // as kTile (and in its order), four k-steps at a time
    kPerWave,   // a tile (pair) per wave, rows read where they lie
};

// Where rows are read where they lie, a block whose eight waves have all of their k-steps under way has its compute unit to itself;
// four steps at a time, two such blocks share one, and 32 rows are one block and not two.  us at once / in fours: 7 rows of 2240 to 1008
// columns 3.7 / 4.1, 11 of 2752 to 11 920 10.3 / 11.5, 49 of 2560 to 12 608 32.7 / 55.5; seven and eight steps a wave are two trips of four: 5
// of 3136 to 2272 4.5 / 4.3, 2 of 3712 to 8528 8.3 / 7.8, but 31 of 3200 to 800 6.2 / 8.9 and 40 of 3456 to 9792 28.2 / 37.7; 21 of 4288 to
// 12 016 29.8 / 28.5, SwiGLU of 18 of 4288 to 7408 28.7 / 21.5, of 48 of 4864 to 1376 16.3 / 22.7, of 33 of 4800 to 3504 21.9 / 20.5.
inline bool long_tile_pays(const W8Product &p, int compute_units) {
    const int share = p.share(), rt = p.row_tiles();
    if (share <= 6) return true;
    if (rt == 1) return share >= 9 && !p.glu && (p.rows > 8 || 4 * p.tiles < 3 * compute_units);
    if (rt == 2) return p.glu ? 2 * p.tiles <= compute_units : 10 * p.tiles <= 6 * compute_units;
    return !p.glu || share == 7 || p.tiles * rt <= 2 * compute_units;
}

inline W8Form choose_w8_form(const W8Product &p, bool normalises, int compute_units) {
    if (p.k <= kRowsMaxK) {
        if (!rows_take_split(p, compute_units)) return rows_fit_lds(p) ? W8Form::kRowsInLds : W8Form::kPerWave;
        // A few long rows are not worth their way through LDS (us where they lie / so; four k-steps a wave are one trip of kSplit as well, which
        // is the quicker one while every block has a compute unit: 1 row of 2048 to 3040 columns 3.5 / 3.7, SwiGLU of 9 of 1664 to 256
        // 3.7 / 4.3, but 8 of 2048 to 896 3.5 / 3.2; with more blocks, SwiGLU of 1 of 1728 to 9152 8.1 and 9.1 / 8.5, 2 of 1856 to 11 696 5.7
        // and 6.1 / 6.3).
        if (!normalises && p.share() == 4) {
            if (p.tiles <= compute_units && p.rows <= (p.glu ? 16 : 4)) return W8Form::kSplit;
            if (p.rows <= 4 && 2 * (p.glu ? 2 : 1) * p.tiles > 5 * compute_units) return W8Form::kTileLong;
        }
        return W8Form::kTile;
    }
    if (p.tiles >= 4 * compute_units) return W8Form::kPerWave;
    if (normalises || p.k > kTileMaxK) return W8Form::kSplit;
    if (sums_in_pairs(p, compute_units)) return W8Form::kSmallTile;
    return long_tile_pays(p, compute_units) ? W8Form::kTileLong : W8Form::kSplit;
}

} // namespace nnhip
