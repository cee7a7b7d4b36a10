// How a dense layer is packed where more than one kernel computes it: plain host arithmetic, so that a test can hold the choice
// against the measured times without a device.
#pragma once

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

} // namespace nnhip
