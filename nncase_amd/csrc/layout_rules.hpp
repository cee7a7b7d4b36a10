// Which kernel a layout operator takes where more than one moves it: plain host arithmetic, so that a test can hold the choice
// against the measured times without a device.  Elements, bytes and tiles are weighed per compute unit.
#pragma once

#include <algorithm>
#include <cstdint>

namespace nnhip {

// Whether pack / unpack of rows that are no whole dwords goes through the tile kernel (true) or takes a thread per element.  A
// tile's load, barrier and store take 3.5 to 5 us however few tiles there are, a thread per element 2.5 to 3 and then some 7
// us per million elements of the packed tensor (packing), or 3 per million of the plain one and a little for the packed lines it
// picks them from (unpacking: runs below 16 bytes pick neighbours from a line that is there already).
// us, per element / tiles: pack of u8 155 x 19 x 19 by 32 3.3 / 4.1, 75 x 51 x 51 by 32 4.5 / 4.2, 155 x 75 x 75 by 4 9.0 / 4.4;
// unpack of u8 155 x 51 x 51 by 32 3.4 / 3.5, 155 x 75 x 75 4.8 / 3.6, by 4 4.6 / 4.9; of float16 155 x 75 x 75 by 4 5.6 / 5.1.
inline bool ragged_tile_pays(int es, uint32_t la, uint64_t plain, uint64_t packed, bool pack, int compute_units) {
    if (pack) return packed >= 640ull * compute_units;
    return plain + packed / 8 >= (la * es >= 16 ? 1880ull : la * es >= 8 ? 3200ull : 3840ull) * compute_units;
}
// Whether packing reads rows of whole dwords, but not of whole 16-byte pieces, in unaligned pieces and the smaller tiles (true) or
// dword by dword.  us, dwords / pieces: u8 75 x 38 x 38 by 32 5.9 / 4.1, float32 155 x 51 x 51 by 32 6.4 / 4.5; but 4 lanes of
// float16 8 x 155 x 150 x 150 28.2 / 35.9, a lane group of less than a tile, u8 75 x 14 x 14 by 16, 3.7 / 4.0, and past 16 MB,
// where it is all memory traffic, float32 4 x 155 x 201 x 201 by 32 49.6 / 52.9.
inline bool unaligned_pieces_pay(uint32_t la, uint64_t row_bytes, uint64_t plain_bytes) {
    return la >= 16 && la * row_bytes >= 12288 && plain_bytes < ((uint64_t)16 << 20);
}
// Whether a relayout whose rows are no whole dwords goes through the tile kernel (true) or through 32 x 32 tiles, by the number
// of the latter per compute unit: they cost 2.4 us and 1 to 2 ns a block from a few thousand blocks on, the tile kernel 4 to 6 us and
// half of that per element or less.  us, 32 x 32 / tiles, both directions: u8 75 x 119 x 119 3.4 3.6 / 6.5 7.8, 155 x 117 x
// 117 5.9 6.3 / 6.0 5.8, 2 x 75 x 151 x 151 7.7 8.1 / 7.1 7.3, 5 x 155 x 151 x 151 23.6 23.8 / 15.1 14.7; float16 75 x 167 x 167 5.4
// 6.6 / 7.6 8.1, 2 x 155 x 151 x 151 13.3 13.3 / 13.5 13.8, 5 x 155 x 151 x 151 37.0 35.9 / 26.8 27.3.  (One to sixteen channels
// leave more than half of every 32 x 32 tile empty: float16 15 x 3 x 151 x 151 7.2 7.8 / 5.1 5.6.)
inline bool ragged_transpose_pays(int es, int batch, int rows, int cols, int compute_units) {
    const uint64_t tiles32 = (uint64_t)batch * ((rows + 31) / 32) * ((cols + 31) / 32);
    return tiles32 >= (es == 1 ? 16ull : std::min(rows, cols) <= 16 ? 24ull : 32ull) * compute_units;
}

} // namespace nnhip
