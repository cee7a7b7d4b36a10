"""How a dense layer of narrow or odd channel counts is packed, held against measured times (us on the device, u8 and float32
outputs): the choice is no more than a fifth slower than the other.  And the output tile of the window kernel against its
definition.  The rules are host arithmetic (csrc/qconv_rules.hpp), compiled here for the CPU."""
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
