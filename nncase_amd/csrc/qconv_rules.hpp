// How a dense layer is packed where more than one kernel computes it, and how its output is cut into tiles: plain host arithmetic,
// so that a test can hold the choices against measured times and against their definition without a device.
#pragma once

#include <algorithm>
#include <cstdint>

namespace nnhip {

// Whether a layer whose channels per group are no multiple of 16 is packed with its taps rounded up to 16 channels, for the
// ragged loader of the wide kernels (true), or as it is, for the small tiles that read pieces of 8 or 4 channels; other channel
// counts have no choice.  The wide kernels need work to fill (a block's set-up takes a microsecond more) and pay for the channels
// they round up by; `pixels`: of the launches to come, 0 = unknown.  us, small tiles / rounded up:
//   * 4 channels, four times the products: 4 -> 8 5x5 stride 2 of 3136 pixels 4.3 / 6.4, 4 -> 6 7x7 of 13 778 5.2 / 8.1, 32 groups of
//     4 -> 4 3x3 of 3136 129 / 171; but single taps (4 -> 81 of 6724 5.4 / 4.6) and small
//     windows with many outputs (4 -> 99 2x2 of 13 068 6.3 / 5.1, 4 -> 113 3x3 of 18 496 10.6 / 7.7)
//   * 8 channels, twice: 8 -> 10 5x5 of 40 432 6.4 / 8.4; no size measured where they win
//   * other multiples of 8 lose a little up to 16 k-steps with few outputs in all (24 -> 32 3x3 stride 2 of 784 pixels 4.3 / 5.3,
//     40 -> 32 4.9 / 6.2; four groups of 24 -> 6 7x7 34.8 / 46.9) and win with more (72 -> 64 3x3 of 25 088 13.4 / 9.3, 24 -> 128
//     of 12 544 7.7 / 6.0)
//   * multiples of 4, whose pieces are half as long, from fewer outputs on (12 -> 32 3x3 stride 2 of 784 pixels 4.4 / 4.9, of 12 544
//     5.3 / 5.3; 12 -> 128 3x3 of 12 544 7.3 / 5.6; 52 -> 32 stride 2 of 784 7.0 / 6.3), and always as single taps (12 -> 64 of 3136
//     4.1 / 3.5)
// (Of 750 layers of 4 to 88 channels the choice loses more than 5 % to the small tiles on 22, a fifth at most.)
inline bool ragged_pays(int g_ic, int taps, int g_oc, int64_t pixels) {
    if (g_ic % 4 != 0) return true;
    if (g_ic == 4) return taps == 1 || (taps <= 4 && (g_oc >= 64 || pixels >= 32768)) || (taps <= 9 && g_oc >= 64 && pixels >= 8000);
    if (g_ic == 8) return false;
    const int ksteps = (taps * ((g_ic + 15) / 16 * 16) + 63) / 64;
    const int64_t outputs = pixels * g_oc;
    if (pixels <= 0) return ksteps >= 5 || g_ic % 8 != 0;
    if (g_ic % 8 == 0 && g_oc < 16 && pixels < 32768 && ksteps < 34) return false;
    if (ksteps >= 17) return true;
    if (g_ic % 8 == 0) return ksteps >= 5 && (outputs >= 200000 || pixels >= 32768);
    return g_ic > 48 || taps == 1 || outputs >= 70000 || pixels >= 6000;
}

// Whether a reduction of two to four k-steps (of 64) whose channels are whole 16-channel slices takes the small wide blocks and not
// the small tiles; longer ones always do, one k-step never.  `tiles`: the 16-channel tiles per chunk that the small tiles would be
// packed with.  Those write a chunk whose lanes (a quarter of it each) all hold real channels with their short epilogue, and then are
// the quicker ones whatever the size (205 209 pixels 128 -> 128 1x1 13.4 us, wide blocks 19.1; 154 568 of 256 -> 192 23.5 / 29.7;
// 12 544 of 96 -> 576 6.4 / 7.1); with other channel counts their stores are piecemeal, where the wide blocks write whole rows: us,
// small tiles / wide blocks, by tiles
//   * 4 and fewer: a tenth quicker on the small tiles in the mean, 357 309 pixels 80 -> 45 1x1 20.0 / 27.4
//   * 5 and 6: a tenth slower, 9464 pixels 112 -> 321 to floats 10.2 / 8.1
//   * 8 and more: a quarter slower, 54 450 pixels 192 -> 224 1x1 24.9 / 12.1, 32 768 rows 192 -> 1000 34.7 / 26.8, 102 400 pixels
//     128 -> 255 44.4 / 28.8
// (Float32 results, of which a layer's weights know nothing when they are packed, would take the wide blocks in whole chunks too:
// 40 095 pixels 128 -> 320 23.1 / 16.9.  Of 1350 such layers, a quarter of them to floats, the choice is 1.3 % off the quicker one in the
// mean and loses more than 5 % to the small tiles on 13, 16 % at most.)
inline bool small_wide_pays(int g_oc, int ksteps, int tiles) {
    return ksteps >= 5 || (ksteps >= 2 && tiles >= 5 && g_oc % (4 * tiles) != 0);
}

// Rows per block, in sixteens of a wave (a block is four waves of them high: 2, 3 or 4 stand for 128, 192 and 256 rows), of the
// products that the kernel of 256-channel chunks fed by DMA alone computes.  A block has its compute unit to itself, so a launch is
// rounds of the device, each a fill and an epilogue (8.5 us; 12.5 with the stores of 256 x 256 outputs) and the k-steps (0.52, 0.80
// and 0.97 us of 64 at 128, 192 and 256 rows: more rows share a k-step's weights).  us at 128 / 192 / 256 rows: 5000 rows of 3000 to
// 2100 columns 59.6 / 46.2 / 53.7 (360, 243 and 180 blocks), 4096 of 3008 to 2048 32.4 / 38.6 / 45.2, 32 768 of 1024 to 1024
// 67.0 / 65.7 / 56.0, 10 000 of 640 to 2000 37.8 / 36.3 / 42.7, 16 000 of 2048 to 512 25.0 / 29.5 / 35.5.
struct DmaRows {
    int rg;
    double us;
};
inline DmaRows choose_dma_rows(int64_t rows, int nchunks, int ksteps, int compute_units) {
    constexpr double outside[3] = {8.5, 8.5, 12.5}, per_kstep[3] = {0.52, 0.80, 0.97};
    DmaRows best{0, 0};
    for (int rg = 4; rg >= 2; rg--) {
        const int64_t blocks = (rows + rg * 64 - 1) / (rg * 64) * nchunks, rounds = (blocks + compute_units - 1) / compute_units;
        const double us = rounds * (outside[rg - 2] + ksteps * per_kstep[rg - 2]);
        if (!best.rg || us < best.us) best = {rg, us};
    }
    return best;
}

// Whether a product takes that kernel and not blocks of 128 channels and fewer: with a 256 x 256 block for more than half of the
// compute units, or where its rounds are quicker than what the others reach (1.05 POP/s behind 4 us).  us, the others / it: 4096 rows
// of 3008 to 2048 40.9 / 32.4, 1300 of 4096 to 4096 44.3 / 31.6, 3680 of 2156 to 1554 35.0 / 24.9; but 5996 of 2816 to 624
// 21.3 / 25.4, 8520 of 1032 to 377 12.8 / 16.1, 1532 of 704 to 3941 12.2 / 13.2.
inline bool dma_pays(int64_t rows, int n, int ksteps, int compute_units) {
    if (n <= 128) return false;
    const int nchunks = (n + 255) / 256;
    if (2 * ((rows + 255) / 256) * nchunks > compute_units) return true;
    return choose_dma_rows(rows, nchunks, ksteps, compute_units).us < 4 + 2.0 * (double)rows * n * ksteps * 64 / 1.05e9;
}

// How a pair of dense 1x1 convolutions (k1 -> n1 -> n2 channels) is launched: a wave per channel tile of whichever convolution has more of
// them in a workgroup (up to the variant's most), and enough workgroups to occupy the device: pixel tiles x ranges of the second
// convolution's channel tiles.  With a depthwise stage, also enough threads that none of them walks more than four of the 16 pixels,
// and tiles of 8 or 4 pixels where that still leaves a compute unit to every workgroup.
struct PairSplit {
    int ranges, tiles_per_block, waves;
    int pixels; // of a workgroup
    bool once;  // no wave has a second tile or chunk of its reduction to come
    bool small; // the variant for short reductions
    bool apart; // not as a pair at all, but as two launches of the kernel for one convolution over few pixels
};
inline PairSplit split_pair(int64_t pixels, int k1, int n1, int n2, bool dw, int compute_units) {
    auto up = [](int64_t v, int64_t d) { return (int)((v + d - 1) / d); };
    const int ks1 = up(k1, 64), ks2 = up(n1, 64), t1 = up(n1, 16), t2 = up(n2, 16);
    PairSplit s;
    s.small = ks1 <= 4 && ks2 <= 2;
    const int max_waves = s.small ? 16 : 12;
    int ptiles = 0;
    auto tile = [&](int pt) {
        s.pixels = pt, ptiles = up(std::max<int64_t>(pixels, 1), pt);
        const int want = ptiles >= 512 ? 1 : 512 / ptiles;
        s.tiles_per_block = up(t2, std::min(up(t2, max_waves), want));
        s.ranges = up(t2, s.tiles_per_block);
        s.waves = std::min(max_waves, std::max(t1, s.tiles_per_block));
        if (dw) s.waves = std::min(max_waves, std::max(s.waves, up((int64_t)k1 * pt, pt == 16 ? 1024 : 256)));
        s.once = t1 <= s.waves && s.tiles_per_block <= s.waves && ks1 <= 16 && ks2 <= 4;
    };
    tile(16);
    if (dw)
        for (int pt = 4; pt < 16; pt *= 2) {
            tile(pt);
            if (s.once && (int64_t)ptiles * s.ranges <= compute_units) break;
            tile(16);
        }
    // ... but no more than lets every workgroup be resident at once (a second round of workgroups doubles the
    // launch's latency chain; a wave that takes two channel tiles one after the other adds a fraction of it)
    const int occupancy = s.small ? 4 : 3; // waves per SIMD the variant is built for
    s.waves = std::max(1, std::min(s.waves, 4 * occupancy / std::max(up((int64_t)ptiles * s.ranges, compute_units), 1)));
    s.once = s.once && t1 <= s.waves && s.tiles_per_block <= s.waves;
    // With more tiles between the two than a workgroup has waves, some waves take several tiles of the whole reduction, chunk by chunk:
    // so many trips to the weights in turn.  Apart where they are many, three tiles of few pixels, or more workgroups than units (us in a
    // chain, pair / apart: 49 pixels 960 -> 320 -> 1280, 6 trips, 8.4 / 7.3; 50 of 960 -> 512 -> 96, 8, 10.0 / 7.0; 57 of 448 -> 480 -> 512, 3
    // tiles, 7.6 / 6.7; 1143 of 640 -> 208 -> 640, two workgroups a unit, 14.9 / 8.7; but 60 of 512 -> 240 -> 1280, 3, 5.8 / 6.8, 85 of 384 ->
    // 288 -> 64, 4, 5.8 / 6.9, 492 of 640 -> 240 -> 256, 5, 7.2 / 8.0, 585 of 320 -> 416 -> 24, 3 tiles, 6.5 / 7.2, 961 of 576 -> 272 -> 96, 6,
    // 7.9 / 8.8).  Up to the pixels for which the kernel of few is measured: 3136 of 512 -> 256 -> 512 13.0 / 14.1.
    const int tiles1 = up(t1, s.waves), tiles2 = up(s.tiles_per_block, s.waves), trips = tiles1 * up(ks1, 8) + tiles2 * up(ks2, 4);
    s.apart = !dw && !s.small && t1 > max_waves && n1 % 16 == 0 && pixels <= 1600 && // (whose rows are whole pieces)
              (trips >= (pixels <= 800 ? 6 : 7) || (tiles1 >= 3 && pixels <= 128) || tiles2 >= 2);
    return s;
}

// The tile of at most `pix` output pixels (32 at most side by side) that covers an out_h x out_w image in the fewest blocks, rows
// and columns spread evenly over them; among equals the one with the smallest input, among those the widest (below four columns
// the first that does no better ends the search).  span: what a window reads, its dilation included.  (Asked for on every launch,
// so it goes through tile widths, 32 at most, and not through all numbers of tiles side by side: 0.7 -> 0.3 us for rows of 320
// pixels, 2.1 -> 0.35 for 1280.)
struct OutputTile {
    int th, tw;         // output pixels
    int across, down;   // tiles per image
    int in_rows, in_cols;
};
inline OutputTile choose_output_tile(int out_h, int out_w, int pix, int stride_h, int stride_w, int span_h, int span_w) {
    OutputTile best{};
    long long best_blocks = -1, best_area = 0;
    for (int tw = std::min({out_w, pix, 32}); tw >= 1; tw--) {
        const int across = (out_w + tw - 1) / tw;
        if ((out_w + across - 1) / across != tw) continue; // (as many tiles of fewer columns each)
        const int rows = std::min(pix / tw, out_h);
        const int down = (out_h + rows - 1) / rows, th = (out_h + down - 1) / down;
        const int in_rows = (th - 1) * stride_h + span_h, in_cols = (tw - 1) * stride_w + span_w;
        const long long blocks = (long long)across * down, area = (long long)in_rows * in_cols;
        if (best_blocks >= 0 && (blocks > best_blocks || (blocks == best_blocks && area >= best_area))) {
            if (tw < 4) break;
            continue;
        }
        best_blocks = blocks, best_area = area;
        best = OutputTile{th, tw, across, down, in_rows, in_cols};
    }
    return best;
}

// A division of what counts the window kernel's threads or pixels, two instructions: p / d = p * mul >> 20 for 0 <= p < kTileDivMost and
// every d >= 1.  (mul is less than 1 above 2^20 / d, so the product less than p above 2^20 p / d: short of the next whole number while
// p d < 2^20, and of the first while p < d, which covers every larger d.)
constexpr int kTileDivMost = 1024;
inline uint32_t make_tile_div(int d) { return ((1u << 20) + (uint32_t)d - 1) / (uint32_t)d; }

// Whether a launch of the window kernel as planned is quicker than the implicit GEMM of the same layer (byte results, strides of 1
// and 2, whole_window_ksteps and more).  us, implicit GEMM / window kernel:
//   * tiles that images do not fill by half stay, their surplus pixels are multiplied and dropped; with fewer than three waves per
//     compute unit a sixth is too much (3388 pixels 256 -> 170 in two groups, 63 % full, 12.1 / 14.4)
//   * with fewer than three waves per two compute units (stride 2: four per unit) the k-steps split over groups of waves win, in the
//     ring and, quicker still, here (split_window_pays)
//     (400 pixels 256 -> 256 7.1 / 7.5; 1600 pixels 128 -> 256 stride 2 5.8 / 6.8)
//   * blocks of two waves have to leave room in LDS for four of a compute unit from 400 channels on (560 -> 32 3x3 of 40 344 pixels
//     27.4 / 34.2, 512 -> 48 5x5 of 18 150 41.9 / 49.0; up to there three are enough: 256 -> 32 5x5 of 85 264 61.4 / 43.6), and for
//     five with stride 2, whose staging is four times as long (400 -> 320 of 11 664 33.8 / 55.4, 128 -> 32 of 147 456 28.7 / 57.1);
//     blocks of 128 pixels at stride 1 win with what fits (80 -> 32 5x5 of 149 187 37.9 / 19.0), blocks of eight waves with one
//     per compute unit (128 -> 128 7x7 stride 2 of 56 448 78.5 / 55.7)
//   * 32 pixels per block do not pay for the staging of less than five k-steps (22 445 pixels 16 -> 128 3x3 in two groups 8.4 / 10.8,
//     64 -> 64 2x2 of 35 301 4.6 / 5.9, 16 -> 64 3x3 of 287 296 11.9 / 17.3), and are too few where a short reduction meets a launch
//     many times what the device holds: 64 -> 64 of 421 362 39.0 / 46.2, 32 -> 316 of 104 907 36.6 / 40.1 (but 64 -> 64 of 102 400
//     12.7 / 11.5)
// (Of 660 launches planned here, of windows over 1000 to 700 000 pixels, the choice is 1.1 % off the quicker one in the mean and
// loses more than 5 % to the implicit GEMM on 44, 30 % at most.)
struct TileLaunch {
    int stride_w, ksteps;
    int channels;   // of a group's input
    int pix, waves; // per block
    size_t lds;
    long long tiles, chunks, pixels;
};
inline bool tile_kernel_pays(const TileLaunch &l, int compute_units) {
    const long long launched = l.tiles * l.chunks * l.waves, room = l.tiles * l.pix;
    if (l.lds > 160 * 1024 || 2 * l.pixels < room) return false;
    if (2 * launched < (l.stride_w == 2 ? 8 : 3) * (long long)compute_units) return false;
    if (launched < 3 * (long long)compute_units && 20 * l.pixels < 17 * room) return false;
    if (l.waves > 2) return true;
    const size_t resident = 160 * 1024 / l.lds;
    if (l.stride_w == 2 && resident < 5) return false;
    if (l.pix < 128 && l.channels > 400 && resident < 4) return false;
    return l.pix > 32 || (l.ksteps >= 5 && launched <= 9ll * l.ksteps * compute_units);
}

// The k-steps from which the window kernel's undivided blocks are worth their staging; fewer are the epilogue's work alone.  `tiles`: of 16
// channels, packed together; eight take blocks of eight waves.  us, implicit GEMM or ring / window kernel:
//   * stride 1: three (16 -> 32 3x3 of 1 638 400 pixels 41.4 / 36.7; two, 802 816 pixels 16 -> 32 2x2, 14.9 / 18.6)
//   * stride 2 brings in four times the input: five (32 -> 64 3x3 of 25 600 5.6 / 4.7, 32 -> 131 of 7605 6.1 / 5.1; three, 16 -> 142 of 8192
//     4.7 / 5.4), eight tiles seven (33 -> 67 of 14 112 7.0 / 5.7, 64 -> 128 of 25 600 8.3 / 7.1; five, 32 -> 214 of 22 472 8.5 / 9.7)
//   * channels that are no multiple of 16, eight tiles and stride 1: nine (35 -> 106 3x3 of 64 800, seven, 14.2 / 16.1; 111 -> 319 of 25 392
//     35.6 / 20.6)
inline int whole_window_ksteps(int stride_w, int tiles, bool ragged) {
    if (stride_w == 2) return tiles == 8 ? 7 : 5;
    return ragged && tiles == 8 ? 9 : 3;
}

// Whether groups of waves that share a block's k-steps (TileLaunch::waves counts all of them) are quicker in the window kernel than
// whatever else the layer would take: all blocks run at once, with no more than eight waves to a compute unit, of which at least four
// come from what fits into its LDS side by side.  us, without / with: 128 -> 128 3x3 of 1600 pixels 5.3 / 4.0, 256 -> 256 of 400 6.8 / 4.7,
// 512 -> 512 of 400 11.0 / 7.9, 64 -> 64 of 1600 4.5 / 3.8, 256 -> 24 7x7 of 1083 24.3 / 7.8, 32 -> 32 of 6400 4.2 / 3.5; past eight waves
// 80 -> 32 of 51 200 5.6 / 6.1, 128 -> 160 of 12 288 8.2 / 8.9; too few side by side 512 -> 160 stride 2 of 1352 12.1 / 14.0.
// (Of 338 launches of 60 to 60 000 pixels 1.37 times as quick in the mean, 1.2 % off the quickest of all shapes.)
inline long long split_window_waves(int compute_units) { return 8ll * compute_units; }
inline bool split_window_pays(const TileLaunch &l, int compute_units) {
    if (l.lds > 160 * 1024) return false;
    const long long blocks = l.tiles * l.chunks, resident = (long long)(160 * 1024 / l.lds);
    return blocks * l.waves <= split_window_waves(compute_units) && blocks <= resident * compute_units && resident * l.waves >= 4;
}

// Whether two dense 1x1 convolutions, the second over the first one's result, are quicker as a pair than as two launches: while every
// workgroup has a compute unit to itself, or several share one and each requests everything at once and repeats nothing (one range), or
// what the workgroups stream between them is little (us of the two / the pair, 20 in a chain, with their depthwise stage where there is
// one, joined where it is: 384 -> 64 -> 384 of 196 pixels 8.9 / 4.6, 576 -> 96 -> 576 of 1200 11.4 / 8.6 and, 300 workgroups, of 1600
// 12.1 / 14.5, 960 -> 160 -> 960 of 588 11.7 / 9.7, 384 -> 64 -> 384 of 2400 9.9 / 12.4; one range 256 -> 128 -> 128 of 6272 8.2 / 4.7, 128 ->
// 64 -> 64 of 12 800 7.0 / 4.6; little 32 -> 16 -> 96 of 12 544 9.6 / 6.9).  Of 1274 such pairs and triples the choice is 0.7 % off the quickest
// of the three in the mean, 43 % at most (32 -> 100 -> 300 of 6400 9.3 / 6.5).
inline bool pair_pays(int64_t pixels, int k1, int n1, int n2, int compute_units) {
    const PairSplit s = split_pair(pixels, k1, n1, n2, false, compute_units);
    const int64_t ptiles = (pixels + 15) / 16, blocks = ptiles * s.ranges;
    if (blocks <= compute_units) return true;
    if (ptiles > 4ll * compute_units) return false;
    return (s.once && s.ranges == 1) || (s.small && ptiles * ((int64_t)k1 * n1 + (int64_t)n1 * n2) <= (4 << 20));
}

// Whether a depthwise stage in front joins the pair's launch: while the plan for it requests everything at once and no thread has more
// than two and a half windows of four channels (us of the two launches / joined, over 20 in a chain: 192 -> 32 -> 192 of 784 pixels
// 6.4 / 4.2, 384 -> 64 -> 384 of 196 6.7 / 4.6, 576 -> 96 -> 576 7.7 / 5.5, 960 -> 160 -> 960 of 49 8.8 / 7.4; 2.5 windows 960 -> 88 -> 912
// of 363 8.4 / 8.0, 2.6 496 -> 8 -> 824 of 576 6.7 / 7.4, 4.2 800 -> 72 -> 928 of 507 8.2 / 10.6; several tiles a wave 592 -> 228 -> 160 of
// 16 10.2 / 11.1, 528 -> 32 -> 812 of 1323 13.8 / 25.6).
inline bool front_pays(int64_t pixels, int k1, int n1, int n2, int compute_units) {
    const PairSplit s = split_pair(pixels, k1, n1, n2, true, compute_units);
    return s.once && 2 * (int64_t)s.pixels * (k1 / 4) <= 5 * (int64_t)s.waves * 64;
}

} // namespace nnhip
