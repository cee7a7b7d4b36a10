"""Which kernel computes a W8A16 product (csrc/w8a16_rules.hpp): held against measured times, and one order of adding for a product
whether its rows are normalised on the way or before.  Host arithmetic, compiled here for the CPU."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nncase_amd", "csrc")
FORMS = ["tile", "tile_long", "small", "rows", "split", "per_wave"]


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("w8")
    (d / "w.cpp").write_text("""#include "w8a16_rules.hpp"
using namespace nnhip;
extern "C" int form(int m, int k, int tiles, int glu, int norm) { return (int)choose_w8_form(W8Product{m, k, tiles, glu != 0}, norm, 256); }
extern "C" int pairs(int m, int k, int tiles, int glu) { return sums_in_pairs(W8Product{m, k, tiles, glu != 0}, 256); }
extern "C" int fit(int m, int k) { return rows_fit_lds(W8Product{m, k, 1, false}); }
""")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "w.cpp"), "-o", str(d / "w.so")])
    return C.CDLL(str(d / "w.so"))


# (rows, k, columns, SwiGLU, normalised, us by each kernel that computes it in the product's order of adding; up to k = 2048 "rows" is another
# order, which the rule may choose for a product)
MEASURED = [
    (6, 384, 16704, 0, 0, dict(tile=4.21, rows=4.17, split=7.43)),
    (2, 768, 13536, 0, 0, dict(tile=4.36, small=13.16, rows=4.99, split=5.53)),
    (4, 1984, 12816, 0, 0, dict(tile=7.11, tile_long=7.35, rows=8.01, split=7.47)),
    (2, 2176, 12256, 0, 0, dict(tile_long=6.85, small=11.27, split=7.31)),
    (6, 3968, 576, 0, 0, dict(tile_long=4.72, small=4.7, split=4.53)),
    (1, 4608, 1152, 0, 0, dict(tile_long=4.52, small=3.97)),
    (11, 128, 3872, 0, 0, dict(tile=2.67, small=10.8, rows=3.17, split=2.63)),
    (9, 960, 14016, 0, 0, dict(tile=5.01, small=29.43, rows=5.6, split=8.06)),
    (9, 1280, 128, 0, 0, dict(tile=3.04, rows=5.07, split=3.17)),
    (9, 2944, 6160, 0, 0, dict(tile_long=6.85, small=15.31, split=7.43)),
    (14, 3648, 3536, 0, 0, dict(tile_long=6.24, small=12.16, split=5.82)),
    (10, 4928, 3968, 0, 0, dict(tile_long=6.31, split=6.64)),
    (22, 320, 15840, 0, 0, dict(tile=5.67, small=60.43, rows=4.41, split=11.93)),
    (21, 832, 1520, 0, 0, dict(tile=2.99, rows=5.09, split=4.18)),
    (17, 2048, 1120, 0, 0, dict(tile=3.75, tile_long=4.7, split=4.58)),
    (27, 2304, 2800, 0, 0, dict(tile_long=7.34, small=17.45, split=8.61)),
    (27, 3840, 2528, 0, 0, dict(tile_long=9.92, small=15.33, split=8.97)),
    (22, 4800, 3760, 0, 0, dict(tile_long=11.25, small=17.57, split=10.79)),
    (62, 256, 5456, 0, 0, dict(tile=4.91, small=58.09, rows=5.02, split=10.52)),
    (43, 896, 3824, 0, 0, dict(tile=4.38, small=30.85, rows=7.71, split=7.46)),
    (39, 1472, 656, 0, 0, dict(tile=3.25, split=7.4)),
    (55, 2560, 6112, 0, 0, dict(tile_long=17.4, small=56.72, split=29.91)),
    (40, 3456, 9792, 0, 0, dict(tile_long=28.16, small=65.66, split=37.61)),
    (33, 4800, 8176, 0, 0, dict(tile_long=31.74, small=50.49, split=32.57)),
    (2, 128, 9408, 1, 0, dict(tile=3.33, rows=4.48, split=3.53)),
    (6, 1024, 64, 1, 0, dict(tile=3.28, rows=5.02, split=3.42)),
    (4, 2048, 1792, 1, 0, dict(tile=4.11, tile_long=4.2, rows=11.03, split=3.92)),
    (8, 2816, 2336, 1, 0, dict(tile_long=5.55, split=5.97)),
    (2, 3200, 3808, 1, 0, dict(tile_long=5.32, split=4.97)),
    (9, 192, 192, 1, 0, dict(tile=2.89, rows=3.69, split=2.85)),
    (15, 704, 7040, 1, 0, dict(tile=3.97, rows=6.6, split=4.44)),
    (9, 1664, 512, 1, 0, dict(tile=4.29, tile_long=4.06, rows=9.54, split=3.74)),
    (9, 3200, 7616, 1, 0, dict(tile_long=6.59, split=6.62)),
    (24, 128, 18016, 1, 0, dict(tile=5.48, rows=4.61, split=6.84)),
    (32, 896, 96, 1, 0, dict(tile=3.44, rows=6.02, split=5.11)),
    (17, 1152, 8896, 1, 0, dict(tile=7.1, rows=10.06, split=7.97)),
    (32, 3072, 960, 1, 0, dict(tile_long=6.39, split=9.88)),
    (19, 3584, 64, 1, 0, dict(tile_long=6.29, split=7.89)),
    (24, 4480, 992, 1, 0, dict(tile_long=8.73, split=11.77)),
    (40, 320, 15840, 1, 0, dict(tile=6.41, rows=7.02, split=13.77)),
    (48, 960, 27776, 1, 0, dict(tile=14.59, rows=11.96, split=36.75)),
    (44, 1216, 15360, 1, 0, dict(tile=11.69, split=17.59)),
    (48, 2560, 6592, 1, 0, dict(tile_long=12.31, split=17.24)),
    (48, 3456, 12000, 1, 0, dict(tile_long=27.82, split=34.1)),
    (48, 4864, 2752, 1, 0, dict(tile_long=16.22, split=22.69)),
    (1, 448, 560, 0, 1, dict(tile=2.5, rows=4.25, split=3.64)),
    (5, 576, 160, 0, 1, dict(tile=2.99, rows=4.72, split=4.03)),
    (6, 1856, 7264, 0, 1, dict(tile=5.75, rows=9.14, split=9.01)),
    (11, 192, 64, 0, 1, dict(tile=3.39, rows=3.78, split=3.57)),
    (11, 768, 192, 0, 1, dict(tile=3.66, rows=5.09, split=4.96)),
    (12, 2048, 9648, 0, 1, dict(tile=9.44, rows=9.53, split=14.56)),
    (21, 448, 11120, 0, 1, dict(tile=6.79, rows=6.57, split=16.77)),
    (25, 960, 10992, 0, 1, dict(tile=9.93, rows=8.57, split=21.37)),
    (20, 1728, 14544, 0, 1, dict(tile=17.53, rows=12.92, split=30.47)),
    (55, 448, 4992, 0, 1, dict(tile=6.46, rows=9.7, split=24.25)),
    (64, 1024, 272, 0, 1, dict(tile=3.75, split=16.88)),
    (33, 1088, 5056, 0, 1, dict(tile=9.99, split=25.92)),
    (8, 448, 32640, 1, 1, dict(tile=5.81, rows=6.73, split=15.68)),
    (2, 960, 14240, 1, 1, dict(tile=5.13, rows=8.28, split=9.16)),
    (2, 1088, 13504, 1, 1, dict(tile=5.87, rows=9.85, split=10.13)),
    (12, 448, 11488, 1, 1, dict(tile=4.86, rows=6.01, split=9.27)),
    (9, 704, 10496, 1, 1, dict(tile=6.39, rows=7.32, split=9.5)),
    (16, 1088, 576, 1, 1, dict(tile=5.01, rows=8.96, split=6.49)),
    (21, 448, 13120, 1, 1, dict(tile=6.35, rows=7.91, split=12.77)),
    (21, 1024, 11968, 1, 1, dict(tile=8.27, rows=10.45, split=15.23)),
    (17, 1408, 7392, 1, 1, dict(tile=7.04, rows=14.05, split=8.85)),
    (33, 448, 1248, 1, 1, dict(tile=4.18, rows=11.16, split=13.82)),
    (48, 896, 1280, 1, 1, dict(tile=4.47, rows=13.81, split=16.89)),
    (33, 1088, 7840, 1, 1, dict(tile=9.1, split=16.29)),
]


@pytest.mark.parametrize("m,k,n,glu,norm,us", MEASURED)
def test_products_take_the_quicker_kernel(rules, m, k, n, glu, norm, us):
    form = FORMS[rules.form(m, k, n // (32 if glu else 16), glu, norm)]
    assert us[form] <= 1.13 * min(us.values()), form


def test_one_order_of_adding(rules):
    """A product and the one that normalises its rows add in the same order, the kernels are asked for what they are built for, and a
    vocabulary head is never a block per tile."""
    orders = {"tile": "split", "tile_long": "split", "split": "split", "small": "pairs", "rows": "whole", "per_wave": "whole"}
    for m in (1, 4, 5, 8, 9, 16, 17, 32, 33, 48, 49, 64):
        for k in list(range(64, 2112, 64)) + [2112, 2560, 2624, 3072, 3136, 4096, 4160, 5120, 5184, 8192]:
            for tiles in (1, 2, 64, 127, 128, 129, 256, 257, 384, 500, 640, 768, 1000, 1023, 1024, 1279, 1280, 1536, 9496):
                for glu in (0, 1):
                    plain, norm = (FORMS[rules.form(m, k, tiles, glu, v)] for v in (0, 1))
                    pairs = rules.pairs(m, k, tiles, glu)
                    assert (orders[plain] == "pairs") == bool(pairs)
                    assert orders[norm] == ("split" if pairs else orders[plain])
                    assert norm in ("tile", "rows", "split", "per_wave") and (norm != "tile" or k <= 2048)
                    assert plain != "tile" or k <= 2048
                    assert plain != "tile_long" or k <= 5120
                    assert plain != "small" or (k <= 5120 and not glu)
                    assert "rows" not in (plain, norm) or rules.fit(m, k)
                    assert tiles < 9496 or orders[plain] == "whole"
