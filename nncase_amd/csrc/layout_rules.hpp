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

// Bytes of both sides up to which a relayout finds them in the memory side's cache of 256 MiB.
constexpr uint64_t kRelayoutCached = 270000000;
// Whether a relayout's runs along A (na elements, nx of them per image) leave in 16-byte pieces (true) or in dwords.  Within the cache
// they do: float16 1 to 22 % quicker, bytes up to 47.  Past it, where the lines that neighbouring tiles share meet in the memory itself,
// it goes either way by the shape, and the dwords' time is seldom far above the pieces', while the pieces' is up to a quarter above the
// dwords': pieces where that was so of whole classes, us dwords / pieces, [na x nx] of 360 to 800 MB:
//   * bytes, short rows of whole pieces: 32 x 784 195 / 172, 128 x 625 117 / 103, 256 x 3136 152 / 147; not long ones (3136 x 256 159 /
//     169, 784 x 512 271 / 281, 256 x 12 544 143 / 146) nor ragged ones (489 x 1936 155 / 189, 253 x 2025 114 / 131, 254 x 3025 188 / 200; but
//     397 x 6084 178 / 158 and 174 x 900 208 / 186)
//   * float16 but for short ragged rows: 5184 x 96 267 / 246, 199 x 2500 274 / 259, 397 x 6084 1.8 % quicker; 87 x 7225 139 / 172, 111 x
//     784 133 / 158, 254 x 3025 142 / 160.
inline bool wide_runs_pay(int es, uint64_t na, uint64_t nx, uint64_t both_bytes) {
    if (both_bytes < kRelayoutCached || es == 4) return true;
    const bool whole = na * es % 16 == 0;
    if (es == 1) return whole && na <= 576 && (na < 128 || nx < 8000);
    return whole || na > 300;
}

} // namespace nnhip
