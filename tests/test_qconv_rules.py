"""How a dense layer of narrow or odd channel counts is packed, held against measured times (us on the device, u8 and float32
outputs): the choice is no more than a fifth slower than the other.  And the output tile of the window kernel against its
definition, and where that kernel is launched.  The rules are host arithmetic (csrc/qconv_rules.hpp), compiled here for the CPU."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nncase_amd", "csrc")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text("""#include "qconv_rules.hpp"
extern "C" int pays(int ic, int taps, int oc, long px) { return nnhip::ragged_pays(ic, taps, oc, px); }
extern "C" void tile(int h, int w, int pix, int sh, int sw, int kh, int kw, int *out) {
    const nnhip::OutputTile t = nnhip::choose_output_tile(h, w, pix, sh, sw, kh, kw);
    out[0] = t.th, out[1] = t.tw, out[2] = t.across, out[3] = t.down, out[4] = t.in_rows, out[5] = t.in_cols;
}
extern "C" int tile_div(int p, int d) { return (int)((uint32_t)p * nnhip::make_tile_div(d) >> 20); }
extern "C" int wide(int oc, int ksteps, int tiles) { return nnhip::small_wide_pays(oc, ksteps, tiles); }
extern "C" int window(int stride, int ksteps, int channels, int pix, int waves, long lds, long tiles, long chunks, long pixels) {
    return nnhip::tile_kernel_pays({stride, ksteps, channels, pix, waves, (size_t)lds, tiles, chunks, pixels}, 256);
}
extern "C" int split_window(long lds, long tiles, long chunks, int waves) {
    return nnhip::split_window_pays({1, 18, 128, 16, waves, (size_t)lds, tiles, chunks, 16 * tiles}, 256);
}
extern "C" int dma_rows(long rows, int nchunks, int ksteps) { return 64 * nnhip::choose_dma_rows(rows, nchunks, ksteps, 256).rg; }
extern "C" int pair_apart(long pixels, int k1, int n1, int n2, int dw) { return nnhip::split_pair(pixels, k1, n1, n2, dw, 256).apart; }
extern "C" int pair_pays(long pixels, int k1, int n1, int n2) { return nnhip::pair_pays(pixels, k1, n1, n2, 256); }
extern "C" int front_pays(long pixels, int k1, int n1, int n2) { return nnhip::front_pays(pixels, k1, n1, n2, 256); }
extern "C" void pair_plan(long pixels, int k1, int n1, int n2, int dw, int *out) {
    const nnhip::PairSplit s = nnhip::split_pair(pixels, k1, n1, n2, dw, 256);
    out[0] = s.pixels, out[1] = s.ranges, out[2] = s.tiles_per_block, out[3] = s.waves, out[4] = s.once, out[5] = s.small;
}
extern "C" int dma(long rows, int n, int ksteps) { return nnhip::dma_pays(rows, n, ksteps, 256); }
""")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-I", CSRC, str(d / "r.cpp"), "-o", str(d / "r.so")])
    lib = C.CDLL(str(d / "r.so"))
    lib.pays.argtypes = [C.c_int, C.c_int, C.c_int, C.c_long]
    return lib


@pytest.fixture(scope="module")
def ragged_pays(rules):
    return rules.pays


# (channels and outputs of a group, window side, output pixels, us by the small tiles, us rounded up to 16 channels per tap)
MEASURED = [
    (4, 4, 3, 1024, 6.8, 9.8),
    (4, 3, 3, 11979, 33.7, 41.4),
    (4, 16, 7, 392, 9.8, 14.3),
    (4, 6, 7, 13778, 5.2, 8.1),
    (4, 45, 1, 9245, 18.2, 14.3),
    (4, 99, 2, 13068, 6.3, 5.1),
    (8, 4, 5, 864, 16.3, 24.2),
    (8, 25, 7, 5184, 40.9, 64.4),
    (8, 5, 7, 35378, 7.7, 11.5),
    (8, 17, 7, 205209, 48.4, 54.5),
    (12, 15, 2, 1849, 7.5, 8.6),
    (12, 3, 5, 4704, 21.8, 24.5),
    (12, 10, 2, 196, 3.8, 4.4),
    (12, 2, 2, 4332, 7.4, 8.5),
    (12, 214, 1, 6498, 6.1, 5.0),
    (12, 20, 2, 43808, 26.7, 20.4),
    (12, 254, 1, 17424, 16.9, 9.5),
    (20, 17, 3, 1452, 4.8, 5.5),
    (20, 6, 5, 343, 13.0, 15.1),
    (20, 6, 3, 12800, 9.8, 11.4),
    (20, 217, 3, 64, 4.8, 5.5),
    (20, 48, 5, 10584, 38.1, 27.7),
    (20, 45, 5, 13456, 23.6, 14.7),
    (20, 58, 7, 22500, 20.7, 14.2),
    (24, 8, 5, 14045, 53.6, 68.0),
    (24, 5, 5, 14884, 24.2, 32.2),
    (24, 6, 3, 7605, 33.9, 43.7),
    (24, 2, 3, 12675, 17.0, 21.4),
    (24, 71, 7, 20808, 19.6, 16.3),
    (24, 119, 3, 34848, 13.8, 9.8),
    (24, 40, 5, 6534, 30.0, 24.9),
    (28, 67, 7, 2352, 12.9, 8.6),
    (28, 40, 3, 100672, 18.1, 14.7),
    (28, 53, 7, 34992, 32.2, 18.6),
    (40, 5, 3, 4761, 19.4, 26.0),
    (40, 80, 7, 75843, 66.5, 53.4),
    (40, 51, 3, 15125, 9.5, 6.0),
    (40, 92, 7, 8712, 29.3, 14.0),
    (56, 8, 5, 15842, 19.6, 23.0),
    (56, 95, 3, 441, 5.6, 6.9),
    (56, 21, 3, 1058, 5.5, 6.6),
    (56, 73, 3, 625, 5.3, 6.5),
    (56, 2, 7, 4205, 30.7, 24.2),
    (56, 12, 7, 20736, 110.9, 64.5),
    (88, 13, 3, 42588, 56.2, 67.4),
    (88, 29, 3, 4356, 57.6, 67.5),
    (88, 5, 3, 588, 6.7, 7.5),
    (88, 3, 3, 1764, 13.3, 15.3),
    (88, 56, 5, 50, 12.6, 8.8),
    (88, 8, 5, 35378, 53.9, 35.5),
    (88, 3, 7, 158400, 590.9, 488.1),
]


@pytest.mark.parametrize("row", MEASURED, ids=lambda r: "%d-%d-%dx%d-%d" % (r[0], r[1], r[2], r[2], r[3]))
def test_packing_takes_the_quicker_kernel(ragged_pays, row):
    ic, oc, k, px, small, ragged = row
    assert (ragged if ragged_pays(ic, k * k, oc, px) else small) <= 1.2 * min(small, ragged)


def test_channel_counts_without_a_choice(ragged_pays):
    for ic in (1, 2, 3, 5, 6, 7, 9, 30, 90, 3001):
        for taps in (1, 9, 49):
            assert ragged_pays(ic, taps, 1, 1) and ragged_pays(ic, taps, 512, 1 << 20)


@pytest.mark.parametrize("pix", [32, 64, 128])
@pytest.mark.parametrize("stride,span", [(1, 3), (2, 3), (1, 7), (2, 5), (1, 2)])
def test_output_tile_is_the_best_of_all_numbers_of_tiles(rules, pix, stride, span):
    """Fewest blocks, then the smallest input, then the widest tile, over every number of tiles side by side; below four columns
    the first that does no better ends the search."""
    up = lambda a, b: -(-a // b)
    got = (C.c_int * 6)()
    for h in (1, 2, 5, 7, 20, 33, 80):
        for w in list(range(1, 70)) + [80, 111, 160, 320, 321, 1000]:
            best = None
            for nx in range(up(w, min(pix, 32)), w + 1):
                tw = up(w, nx)
                rows = min(pix // tw, h)
                th = up(h, up(h, rows))
                across, down, ih, iw = up(w, tw), up(h, th), (th - 1) * stride + span, (tw - 1) * stride + span
                if best is None or (across * down, ih * iw) < best[0]:
                    best = (across * down, ih * iw), [th, tw, across, down, ih, iw]
                elif tw < 4 and tw != best[1][1]:
                    break
            rules.tile(h, w, pix, stride, stride, span, span, got)
            assert list(got) == best[1], (h, w)


def test_division_of_a_tile(rules):
    for d in list(range(1, 1100)) + [4095, 10240, (1 << 20) - 1, 1 << 20, 1 << 24]:
        assert [rules.tile_div(p, d) for p in range(1024)] == [p // d for p in range(1024)], d
    # (24-bit operands, 32-bit product: the largest of both)
    assert 1023 << 20 < 1 << 32 and 1 << 20 < 1 << 24


# windows of a group's channels -> outputs, window side, stride; k-steps; pixels and waves per block, LDS, tiles, chunks, output pixels;
# us by the implicit GEMM, us by the window kernel (all groups)
WINDOWS = [
    (160, 32, 7, 1, 123, 64, 2, 36960, 1040, 1, 63368, 50.0, 37.7),
    (512, 48, 5, 1, 200, 32, 2, 54560, 588, 1, 18150, 41.9, 49.0),
    (624, 54, 3, 1, 88, 32, 2, 39520, 3400, 1, 106097, 109.9, 77.2),
    (256, 32, 5, 1, 100, 64, 2, 43616, 1520, 1, 85264, 61.4, 43.8),
    (384, 128, 7, 1, 294, 32, 2, 62976, 170, 2, 4802, 48.7, 39.3),
    (256, 32, 5, 1, 100, 64, 2, 41168, 1512, 1, 95256, 64.3, 43.1),
    (192, 22, 7, 1, 147, 64, 2, 46704, 660, 1, 38720, 43.9, 28.1),
    (16, 128, 3, 1, 3, 32, 2, 3280, 765, 2, 22445, 8.4, 10.8),
    (32, 316, 3, 1, 5, 32, 2, 5600, 3366, 5, 104907, 36.6, 40.1),
    (336, 448, 3, 1, 48, 128, 8, 62560, 150, 4, 19200, 60.3, 39.9),
    (384, 224, 5, 1, 150, 128, 8, 99712, 96, 2, 11907, 57.0, 37.9),
    (80, 128, 3, 1, 12, 128, 8, 19936, 512, 1, 59168, 16.1, 12.1),
    (64, 128, 5, 1, 25, 128, 8, 21072, 490, 1, 60025, 25.1, 20.9),
    (80, 32, 5, 1, 32, 128, 2, 20640, 1176, 1, 149187, 37.9, 19.0),
    (112, 32, 5, 1, 44, 128, 2, 29632, 4920, 1, 605160, 163.4, 84.0),
    (96, 32, 3, 1, 14, 128, 2, 24000, 4620, 1, 570288, 62.2, 37.9),
    (16, 18, 5, 1, 7, 128, 2, 7184, 2210, 1, 271445, 39.9, 28.4),
    (16, 64, 3, 1, 3, 32, 2, 3280, 9248, 1, 287296, 23.8, 34.5),
    (16, 64, 3, 1, 3, 32, 2, 3280, 5082, 1, 155232, 15.9, 21.3),
    (528, 320, 3, 1, 75, 32, 2, 33552, 56, 5, 1444, 11.8, 14.5),
    (240, 46, 5, 1, 94, 32, 2, 23296, 270, 1, 6615, 13.6, 16.4),
    (64, 64, 3, 1, 9, 32, 2, 8736, 13770, 1, 421362, 39.0, 46.2),
    (16, 149, 3, 1, 3, 32, 2, 3280, 1386, 3, 36982, 20.0, 23.7),
    (128, 64, 3, 1, 18, 32, 2, 9600, 1058, 1, 33856, 12.0, 8.6),
    (80, 64, 3, 1, 12, 32, 2, 6624, 2310, 1, 71148, 13.4, 9.7),
    (32, 320, 3, 1, 5, 32, 2, 3440, 168, 5, 4356, 6.0, 4.8),
    (16, 48, 7, 1, 13, 32, 2, 3440, 322, 1, 9522, 6.1, 5.2),
    (32, 240, 7, 1, 25, 64, 8, 12256, 84, 2, 4332, 9.5, 7.0),
    (96, 255, 7, 1, 74, 64, 8, 28448, 119, 2, 6800, 21.2, 16.4),
    (192, 128, 3, 1, 27, 64, 8, 22288, 180, 1, 9680, 10.4, 8.7),
    (80, 208, 3, 1, 12, 64, 8, 10464, 84, 2, 4375, 7.1, 6.2),
    (528, 96, 2, 1, 33, 64, 2, 35520, 90, 3, 4320, 7.9, 11.5),
    (304, 16, 3, 1, 43, 64, 2, 28112, 264, 1, 14256, 8.9, 11.8),
    (560, 32, 3, 1, 79, 64, 2, 66336, 672, 1, 40344, 27.4, 34.2),
    (128, 85, 3, 1, 18, 64, 2, 12192, 84, 3, 3388, 12.1, 14.4),
    (528, 16, 2, 1, 33, 64, 2, 43440, 360, 1, 18750, 10.6, 12.4),
    (512, 32, 3, 1, 72, 64, 2, 52512, 225, 1, 12615, 12.3, 14.4),
    (80, 22, 5, 1, 32, 64, 2, 13984, 945, 1, 56307, 33.9, 21.5),
    (16, 15, 7, 1, 13, 64, 2, 4768, 880, 1, 53138, 9.6, 6.5),
    (32, 32, 3, 1, 5, 64, 2, 5504, 663, 1, 39675, 5.9, 4.9),
    (96, 32, 5, 1, 38, 64, 2, 17408, 363, 1, 21675, 11.4, 10.1),
    (48, 272, 7, 2, 37, 128, 8, 38192, 208, 3, 21866, 49.9, 32.5),
    (64, 256, 7, 2, 49, 128, 8, 65936, 108, 2, 13254, 24.0, 16.9),
    (64, 128, 7, 2, 49, 128, 8, 67376, 672, 1, 84672, 59.1, 44.7),
    (192, 512, 3, 2, 27, 128, 8, 121968, 48, 4, 6144, 15.8, 13.2),
    (128, 32, 3, 2, 18, 128, 2, 84448, 1152, 1, 147456, 28.7, 57.0),
    (400, 320, 3, 2, 57, 32, 2, 66384, 405, 5, 11664, 33.8, 55.4),
    (432, 48, 3, 2, 61, 32, 2, 71632, 612, 1, 17956, 19.2, 29.1),
    (288, 48, 3, 2, 41, 32, 2, 48144, 1071, 1, 29988, 16.3, 24.6),
    (192, 184, 3, 2, 27, 32, 2, 33136, 1071, 3, 29988, 25.0, 34.1),
    (368, 128, 2, 2, 23, 32, 2, 45200, 266, 2, 6859, 8.7, 11.9),
    (288, 64, 5, 2, 113, 32, 2, 69360, 720, 1, 23040, 29.4, 39.4),
    (32, 448, 7, 2, 25, 32, 2, 14800, 198, 7, 5808, 15.8, 12.1),
    (48, 448, 5, 2, 19, 32, 2, 10480, 108, 7, 2601, 9.4, 7.5),
    (160, 64, 3, 2, 23, 32, 2, 30960, 1950, 1, 60840, 18.6, 20.9),
    (224, 480, 3, 2, 32, 64, 8, 63968, 60, 4, 3240, 12.2, 10.0),
    (368, 128, 5, 2, 144, 64, 8, 143200, 196, 1, 11881, 33.1, 27.5),
    (128, 96, 3, 2, 18, 64, 8, 45696, 224, 1, 13778, 8.5, 7.5),
    (240, 208, 5, 2, 94, 64, 2, 75616, 92, 7, 3887, 22.8, 38.0),
    (288, 32, 2, 2, 18, 64, 2, 78784, 833, 1, 51425, 15.5, 24.9),
    (192, 32, 7, 2, 147, 64, 2, 105776, 1380, 1, 82810, 101.9, 131.3),
    (112, 16, 3, 2, 16, 64, 2, 32960, 540, 1, 32400, 7.7, 8.7),
]


@pytest.mark.parametrize("row", WINDOWS, ids=lambda r: "%d-%d-%dx%d-s%d-%d" % (r[0], r[1], r[2], r[2], r[3], r[10]))
def test_windows_take_the_quicker_kernel(rules, row):
    ic, oc, k, stride, ksteps, pix, waves, lds, tiles, chunks, pixels, gemm, window = row
    assert (window if rules.window(stride, ksteps, ic, pix, waves, C.c_long(lds), C.c_long(tiles), C.c_long(chunks), C.c_long(pixels)) else gemm) <= 1.2 * min(gemm, window)


def test_window_kernel_is_not_launched_beyond_the_lds(rules):
    args = lambda lds: (1, 40, 256, 128, 8, C.c_long(lds), C.c_long(4000), C.c_long(1), C.c_long(500000))
    assert rules.window(*args(160 * 1024)) and not rules.window(*args(160 * 1024 + 16))


# windows whose k-steps groups of waves share: LDS of a block, tiles, chunks, waves of all groups; us without the split, with it
SPLITS = [
    (16000, 100, 2, 8, 5.28, 4.00),     # 128 -> 128 3x3 of 1600 pixels
    (25000, 28, 4, 8, 6.82, 4.72),      # 256 -> 256 of 400
    (45000, 25, 8, 8, 10.95, 7.91),     # 512 -> 512 of 400
    (22000, 200, 2, 4, 5.79, 5.15),     # 128 -> 128 of 6400, two groups
    (34000, 200, 2, 8, 5.79, 5.50),     # ... four
    (36000, 288, 3, 4, 8.19, 8.86),     # 128 -> 160 of 12 288
    (14000, 1600, 1, 2, 5.60, 6.09),    # 80 -> 32 of 51 200
    (90000, 56, 5, 2, 12.11, 13.99),    # 512 -> 160 stride 2 of 1352: one block of two waves to a compute unit
    (97000, 392, 1, 4, 12.44, 16.40),   # 512 -> 32 stride 2 of 12 544
    (56000, 784, 1, 4, 12.44, 13.87),
]


@pytest.mark.parametrize("row", SPLITS, ids=lambda r: "-".join(map(str, r[:4])))
def test_which_windows_share_their_k_steps(rules, row):
    lds, tiles, chunks, waves, without, split = row
    assert (split if rules.split_window(C.c_long(lds), C.c_long(tiles), C.c_long(chunks), waves) else without) <= 1.1 * min(without, split)
    assert not rules.split_window(C.c_long(160 * 1024 + 1), C.c_long(1), C.c_long(1), waves)


# a group's channels -> outputs, window side, k-steps, the small tiles' 16-channel tiles per chunk, output pixels; us by the small tiles,
# us by the small wide blocks (all groups)
SHORT = [
    (32, 160, 2, 2, 5, 21780, 4.7, 6.7),
    (96, 176, 1, 2, 4, 12943, 3.7, 5.2),
    (112, 176, 1, 2, 4, 14700, 3.8, 5.3),
    (128, 192, 1, 2, 6, 20736, 4.8, 6.3),
    (128, 64, 1, 2, 1, 1377, 2.8, 3.4),
    (128, 96, 1, 2, 1, 2057, 3.3, 3.9),
    (96, 128, 1, 2, 8, 218295, 12.8, 20.4),
    (80, 160, 1, 2, 10, 198450, 16.2, 25.4),
    (128, 144, 1, 2, 9, 139240, 12.3, 19.2),
    (128, 160, 1, 2, 10, 105800, 10.7, 14.5),
    (112, 640, 1, 2, 8, 7200, 4.8, 6.1),
    (80, 576, 1, 2, 12, 34225, 12.7, 15.2),
    (96, 256, 1, 2, 6, 15300, 6.7, 5.5),
    (128, 512, 1, 2, 6, 7943, 6.7, 5.5),
    (80, 560, 1, 2, 6, 6125, 6.4, 5.4),
    (112, 416, 1, 2, 6, 7056, 6.2, 5.4),
    (80, 640, 1, 2, 6, 6292, 6.6, 5.8),
    (112, 176, 1, 2, 12, 35721, 13.2, 7.0),
    (80, 176, 1, 2, 12, 166617, 38.6, 21.0),
    (128, 176, 1, 2, 12, 52272, 17.7, 9.7),
    (128, 416, 1, 2, 16, 42632, 23.0, 15.4),
    (112, 480, 1, 2, 16, 89888, 38.6, 28.6),
    (112, 272, 1, 2, 9, 36288, 12.7, 10.3),
    (160, 96, 1, 3, 6, 86528, 6.8, 10.5),
    (160, 160, 1, 3, 4, 12696, 3.9, 5.6),
    (192, 384, 1, 3, 3, 5400, 4.1, 5.9),
    (16, 64, 3, 3, 4, 49298, 4.9, 6.3),
    (16, 10, 3, 3, 1, 6075, 6.8, 8.3),
    (144, 192, 1, 3, 1, 3042, 3.6, 4.1),
    (176, 144, 1, 3, 9, 230640, 20.4, 34.3),
    (144, 144, 1, 3, 9, 125316, 12.3, 19.0),
    (192, 144, 1, 3, 9, 135036, 13.6, 20.7),
    (160, 128, 1, 3, 8, 259920, 19.5, 25.9),
    (176, 384, 1, 3, 8, 11236, 5.3, 6.4),
    (160, 640, 1, 3, 16, 51005, 27.9, 24.8),
    (16, 256, 3, 3, 6, 15876, 7.5, 5.7),
    (192, 512, 1, 3, 6, 7098, 7.1, 5.8),
    (192, 512, 1, 3, 6, 6724, 7.0, 5.8),
    (144, 512, 1, 3, 6, 6561, 7.0, 5.8),
    (144, 608, 1, 3, 6, 5100, 6.8, 5.7),
    (192, 224, 1, 3, 16, 54450, 24.9, 12.1),
    (160, 208, 1, 3, 16, 58482, 21.8, 12.5),
    (16, 241, 3, 3, 16, 39605, 21.9, 12.7),
    (192, 112, 1, 3, 8, 33489, 9.0, 6.2),
    (16, 406, 3, 3, 16, 20736, 15.6, 11.6),
    (176, 400, 1, 3, 16, 84872, 36.7, 31.0),
    (256, 160, 1, 4, 5, 24548, 5.7, 8.4),
    (240, 128, 1, 4, 4, 16428, 4.1, 5.8),
    (208, 32, 1, 4, 2, 91875, 7.0, 9.8),
    (256, 42, 1, 4, 3, 104976, 25.6, 32.3),
    (256, 189, 1, 4, 2, 6724, 5.2, 6.2),
    (208, 30, 1, 4, 1, 1734, 3.5, 4.0),
    (256, 144, 1, 4, 9, 102900, 12.9, 19.9),
    (240, 128, 1, 4, 8, 204363, 19.0, 27.3),
    (256, 144, 1, 4, 9, 84050, 11.9, 17.0),
    (224, 384, 1, 4, 12, 23805, 8.7, 11.3),
    (256, 192, 1, 4, 12, 81648, 14.2, 17.3),
    (240, 256, 1, 4, 8, 42500, 10.6, 12.2),
    (208, 256, 1, 4, 6, 15488, 7.5, 6.3),
    (256, 512, 1, 4, 6, 7056, 7.3, 6.2),
    (64, 448, 2, 4, 6, 7688, 7.4, 6.4),
    (256, 608, 1, 4, 6, 5202, 7.1, 6.2),
    (224, 176, 1, 4, 12, 36300, 14.8, 9.5),
    (256, 608, 1, 4, 10, 12427, 13.3, 8.7),
    (256, 115, 1, 4, 8, 59290, 13.9, 9.2),
    (224, 512, 1, 4, 12, 25538, 18.5, 13.3),
    (64, 448, 2, 4, 10, 42284, 26.0, 20.4),
    (240, 250, 1, 4, 8, 46656, 18.4, 15.6),
    (128, 255, 1, 2, 16, 102400, 44.4, 28.8),
    (192, 1000, 1, 3, 16, 32768, 34.7, 26.8),
    (144, 24, 1, 3, 2, 200704, 8.9, 10.3),
]


@pytest.mark.parametrize("row", SHORT, ids=lambda r: "%d-%d-%dx%d-%d" % (r[0], r[1], r[2], r[2], r[5]))
def test_short_reductions_take_the_quicker_kernel(rules, row):
    ic, oc, k, ksteps, tiles, pixels, small, wide = row
    assert (wide if rules.wide(oc, ksteps, tiles) else small) <= 1.2 * min(small, wide)


def test_reductions_without_a_choice_of_blocks(rules):
    for oc in (1, 64, 255, 1000):
        assert rules.wide(oc, 5, 1) and not rules.wide(oc, 1, 16)


# rows, reduction, columns, us of the kernel fed by DMA at 256, 192 and 128 rows per block, of blocks of 128 channels and fewer (float32
# results, 256 compute units)
DMA = [
    (5000, 3000, 2100, 53.7, 46.2, 59.6, None),
    (4096, 3008, 2048, 45.2, 38.6, 32.4, 40.9),
    (6000, 1024, 2048, 26.8, 23.5, 29.9, None),
    (1300, 4096, 4096, 54.4, 44.6, 36.1, 47.6),
    (8192, 4096, 1024, 56.1, 47.3, 39.1, 53.8),
    (10000, 640, 2000, 42.7, 36.3, 37.8, None),
    (5000, 512, 4096, 37.2, 32.2, 36.4, None),
    (32768, 1024, 1024, 56.0, 65.7, 67.0, None),
    (20000, 3000, 1500, 108.8, 120.9, 120.7, None),
    (12000, 1000, 700, 29.4, 25.2, 31.1, None),
    (3000, 2048, 3072, 36.8, 31.2, 40.3, None),
    (16000, 2048, 512, 35.5, 29.5, 25.0, 31.9),
    (7000, 2000, 1100, 39.6, 33.1, 43.3, None),
    (25000, 640, 1000, 47.2, 51.6, 49.9, None),
    (2048, 2048, 2048, 33.8, 28.0, 22.1, 19.8),
    (1500, 1500, 3000, 32.4, 26.9, 21.9, 22.8),
    (1000, 4000, 4000, 56.7, 47.2, 38.6, 40.5),
    (3000, 1024, 1024, 22.7, 18.7, 14.4, 13.2),
    (2000, 4000, 1000, 55.2, 44.8, 34.7, 19.9),
    (900, 2000, 2000, 35.1, 28.9, 22.4, 14.2),
]


@pytest.mark.parametrize("row", DMA)
def test_large_products_take_the_quicker_blocks(rules, row):
    rows, k, n = row[:3]
    us = dict(zip((256, 192, 128), row[3:6]))
    rules.dma_rows.argtypes = rules.dma.argtypes = [C.c_long, C.c_int, C.c_int]
    chosen = us[rules.dma_rows(rows, -(-n // 256), -(-k // 64))]
    assert chosen <= 1.06 * min(us.values())
    if row[6] is not None:
        assert (chosen if rules.dma(rows, n, -(-k // 64)) else row[6]) <= 1.06 * min(chosen, row[6])


# (pixels, channels in, between and out, us in a chain as one launch, as two)
PAIRS = [
    (1, 128, 256, 192, 5.16, 5.91), (13, 480, 208, 64, 4.78, 6.48), (60, 512, 240, 1280, 5.79, 6.75), (424, 288, 240, 640, 5.84, 7.62),
    (834, 256, 224, 32, 5.19, 7.21), (73, 480, 288, 32, 5.65, 6.81), (138, 64, 320, 1280, 6.46, 7.11), (1253, 256, 304, 96, 6.27, 8.19),
    (1, 512, 496, 1280, 7.18, 6.14), (57, 448, 480, 512, 7.58, 6.7), (125, 128, 512, 960, 7.62, 6.3), (198, 256, 400, 1536, 7.36, 7.59),
    (86, 640, 240, 128, 6.99, 7.33), (492, 640, 240, 256, 7.15, 8.0), (585, 320, 416, 24, 6.52, 7.23), (892, 192, 256, 960, 11.95, 8.09),
    (1070, 192, 496, 32, 7.05, 7.92), (1, 640, 384, 1280, 8.73, 6.29), (49, 960, 320, 1280, 8.38, 7.26), (122, 640, 384, 320, 9.4, 6.78),
    (692, 1024, 352, 256, 9.03, 8.17), (961, 576, 272, 96, 7.9, 8.77), (819, 192, 288, 1280, 13.88, 10.2), (50, 960, 512, 96, 9.97, 7.03),
    (1143, 640, 208, 640, 14.9, 8.7), (1407, 160, 320, 1280, 16.41, 12.94), (980, 1024, 304, 1280, 19.38, 11.81),
    (3136, 512, 256, 512, 12.97, 14.07), (6400, 960, 320, 320, 23.24, 25.71),
]


@pytest.mark.parametrize("pixels,k1,n1,n2,one,two", PAIRS)
def test_pairs_take_the_quicker_form(rules, pixels, k1, n1, n2, one, two):
    rules.pair_apart.argtypes = [C.c_long, C.c_int, C.c_int, C.c_int, C.c_int]
    assert (two if rules.pair_apart(pixels, k1, n1, n2, 0) else one) <= 1.02 * min(one, two)
    assert not rules.pair_apart(pixels, k1, n1, n2, 1)                         # a depthwise stage in front: always one launch
    assert not rules.pair_apart(pixels, k1, n1 + 4, n2, 0)                      # rows between the two that are no whole pieces


# us of the launches apart / as a pair / with the depthwise stage in the pair's launch (None: no depthwise stage), 20 in a chain
PAIRS_TIMED = [  # (pixels, in, mid, out, ...)
    (392, 32, 16, 96, 7.86, 5.94, 3.53), (6400, 32, 16, 96, 8.57, 6.71, 4.66), (9408, 32, 120, 428, 10.75, 12.41, None),
    (27, 64, 32, 32, 6.06, 3.01, None), (32, 64, 32, 32, 6.13, 3.03, None), (16, 64, 64, 64, 6.46, 2.86, None),
    (800, 64, 64, 64, 5.21, 3.1, None), (6400, 64, 184, 528, 12.14, 18.41, 17.29), (12800, 96, 24, 144, 10.91, 10.24, 9.55),
    (25, 128, 64, 64, 6.35, 3.0, None), (4800, 128, 64, 64, 5.85, 3.55, None), (256, 128, 68, 404, 9.39, 6.66, 4.54),
    (108, 128, 128, 256, 5.45, 4.02, None), (400, 144, 24, 144, 8.88, 6.23, 4.0), (9408, 144, 24, 144, 10.97, 11.3, 12.07),
    (256, 144, 32, 192, 8.17, 6.34, 4.11), (400, 144, 32, 192, 8.38, 6.32, 4.09), (196, 192, 32, 192, 8.38, 6.35, 4.09),
    (6400, 192, 32, 192, 10.12, 9.26, 8.52), (800, 192, 64, 384, 8.75, 6.51, 4.47), (1568, 192, 64, 384, 9.11, 6.74, 5.31),
    (9408, 192, 112, 820, 13.93, 17.61, None), (25, 256, 128, 128, 6.59, 3.43, None), (1600, 256, 128, 128, 6.16, 3.68, None),
    (4704, 304, 76, 1136, 10.2, 19.8, None), (256, 384, 64, 384, 8.69, 6.74, 4.67), (1176, 384, 64, 384, 9.6, 7.17, 6.41),
    (147, 384, 96, 576, 9.07, 7.1, 4.89), (400, 384, 96, 576, 9.39, 7.17, 5.75), (200, 384, 168, 628, 10.0, 7.48, 5.66),
    (100, 416, 196, 56, 6.96, 4.96, None), (200, 448, 188, 200, 7.31, 4.65, None), (200, 480, 152, 92, 6.54, 4.42, None),
    (1200, 496, 12, 448, 6.73, 3.85, None), (392, 512, 256, 256, 7.24, 5.52, None), (4800, 512, 256, 256, 10.17, 12.88, None),
    (588, 528, 64, 340, 6.27, 4.14, None), (100, 544, 64, 92, 9.32, 6.83, 5.12), (400, 576, 96, 576, 10.07, 7.92, 6.79),
    (9408, 576, 96, 576, 17.8, 24.2, 36.94), (100, 576, 160, 960, 10.19, 8.39, 6.25), (4800, 576, 160, 960, 16.21, 28.3, 38.51),
    (3136, 592, 104, 396, 8.26, 12.73, None), (400, 624, 56, 248, 10.07, 7.43, 5.55), (192, 672, 184, 340, 6.94, 5.4, None),
    (196, 704, 160, 816, 6.79, 5.32, None), (3136, 720, 12, 960, 14.56, 19.87, 30.12), (16, 736, 40, 144, 9.34, 6.98, 5.37),
    (300, 736, 40, 456, 6.5, 4.25, None), (49, 736, 108, 1036, 7.19, 4.77, None), (400, 768, 148, 628, 11.36, 8.57, 7.67),
    (392, 768, 164, 832, 11.37, 8.89, 7.94), (4800, 896, 208, 696, 18.02, 28.81, 51.45), (72, 912, 164, 844, 11.18, 8.97, 7.61),
    (18, 944, 124, 100, 10.39, 7.84, 6.82), (196, 960, 64, 332, 6.11, 4.39, None), (400, 960, 160, 960, 10.79, 9.46, 8.97),
    (2352, 960, 160, 960, 13.97, 22.03, 43.51), (9600, 1008, 40, 936, 26.86, 30.01, 50.16), (3200, 1024, 120, 1064, 16.75, 23.29, 45.22),
]


@pytest.mark.parametrize("pixels,k1,n1,n2,apart,pair,joined", PAIRS_TIMED)
def test_pairs_and_fronts_where_they_pay(rules, pixels, k1, n1, n2, apart, pair, joined):
    """At most half more than the quickest of the three as measured (7 in 1000 in the mean of those the rule was drawn from)."""
    for f in (rules.pair_pays, rules.front_pays):
        f.argtypes = [C.c_long, C.c_int, C.c_int, C.c_int]
    as_pair = joined if joined is not None and rules.front_pays(pixels, k1, n1, n2) else pair
    taken = as_pair if rules.pair_pays(pixels, k1, n1, n2) else apart
    assert taken <= 1.5 * min(apart, pair, joined or pair)


def test_pair_plans_cover_the_work(rules):
    """Every channel tile of the second convolution once, a wave per tile where all is requested at once, and small pixel tiles only then."""
    import random
    rng = random.Random(5)
    rules.pair_plan.argtypes = [C.c_long, C.c_int, C.c_int, C.c_int, C.c_int, C.POINTER(C.c_int)]
    out = (C.c_int * 6)()
    for _ in range(20000):
        pixels, k1, n1, n2 = rng.choice([rng.randint(1, 100), rng.randint(1, 20000)]), 16 * rng.randint(1, 64), 4 * rng.randint(1, 128), 4 * rng.randint(1, 400)
        dw = rng.randint(0, 1)
        rules.pair_plan(pixels, k1, n1, n2, dw, out)
        pt, ranges, per, waves, once, small = out
        t1, t2, ks1, ks2 = -(-n1 // 16), -(-n2 // 16), -(-k1 // 64), -(-n1 // 64)
        assert pt in (4, 8, 16) and (pt == 16 or (dw and once)) and (ranges - 1) * per < t2 <= ranges * per
        assert 1 <= waves <= (16 if small else 12)
        if once:
            assert t1 <= waves and per <= waves and ks1 <= 16 and ks2 <= 4 and (not small or (ks1 <= 4 and ks2 <= 2))
