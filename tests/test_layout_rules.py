"""Which kernel a layout operator takes, held against measured times (us on the device, 256 compute units): the choice is never
slower than the other by more than what the two directions of one shape near the crossing differ by.  The rules are host
arithmetic (csrc/layout_rules.hpp), compiled here for the CPU."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nncase_amd", "csrc")
CUS = 256
NEAR = 1.13
SIZE = {"u8": 1, "f16": 2, "f32": 4}


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text("""#include "layout_rules.hpp"
extern "C" int tile(int es, unsigned la, unsigned long plain, unsigned long packed, int pack, int cus) { return nnhip::ragged_tile_pays(es, la, plain, packed, pack, cus); }
extern "C" int pieces(unsigned la, unsigned long row, unsigned long plain) { return nnhip::unaligned_pieces_pay(la, row, plain); }
extern "C" int transpose(int es, int batch, int rows, int cols, int cus) { return nnhip::ragged_transpose_pays(es, batch, rows, cols, cus); }
""")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "r.cpp"), "-o", str(d / "r.so")])
    lib = C.CDLL(str(d / "r.so"))
    lib.tile.argtypes = [C.c_int, C.c_uint, C.c_ulong, C.c_ulong, C.c_int, C.c_int]
    lib.pieces.argtypes = [C.c_uint, C.c_ulong, C.c_ulong]
    return lib


# (type, N, C, H, W, us of NCHW -> NHWC through 32 x 32 tiles, through the tile kernel, us of NHWC -> NCHW likewise)
RELAYOUT = [
    ("u8", 4, 3, 151, 151, 3.2, 3.9, 3.6, 4.6),
    ("f16", 4, 3, 151, 151, 3.2, 3.9, 3.7, 4.6),
    ("u8", 8, 3, 151, 151, 4.2, 4.0, 5.0, 4.6),
    ("f16", 8, 3, 151, 151, 4.4, 4.1, 5.2, 5.0),
    ("u8", 15, 3, 151, 151, 6.1, 4.5, 7.3, 4.8),
    ("f16", 15, 3, 151, 151, 7.2, 4.6, 7.9, 5.8),
    ("u8", 31, 3, 151, 151, 13.1, 5.5, 14.4, 5.7),
    ("f16", 31, 3, 151, 151, 13.7, 6.1, 18.9, 7.5),
    ("u8", 61, 3, 151, 151, 23.8, 8.4, 32.9, 7.5),
    ("f16", 61, 3, 151, 151, 24.3, 9.3, 35.6, 10.6),
    ("u8", 123, 3, 151, 151, 44.8, 14.3, 62.4, 10.0),
    ("f16", 123, 3, 151, 151, 45.7, 13.8, 67.6, 16.4),
    ("u8", 245, 3, 151, 151, 86.4, 23.1, 121.3, 15.7),
    ("f16", 245, 3, 151, 151, 88.0, 22.0, 131.2, 26.3),
    ("u8", 1, 17, 125, 125, 2.5, 3.9, 2.6, 4.7),
    ("f16", 1, 17, 125, 125, 2.6, 3.8, 2.7, 4.7),
    ("u8", 1, 17, 175, 175, 2.7, 3.9, 3.0, 4.7),
    ("f16", 1, 17, 175, 175, 2.7, 4.0, 3.1, 4.9),
    ("u8", 3, 17, 151, 151, 3.7, 4.2, 3.9, 4.9),
    ("f16", 3, 17, 151, 151, 4.6, 4.6, 4.2, 6.1),
    ("u8", 5, 17, 151, 151, 5.3, 4.7, 5.0, 5.8),
    ("f16", 5, 17, 151, 151, 5.4, 5.6, 6.3, 7.2),
    ("u8", 11, 17, 151, 151, 8.8, 7.5, 10.6, 6.9),
    ("f16", 11, 17, 151, 151, 9.3, 9.7, 11.0, 13.3),
    ("u8", 22, 17, 151, 151, 15.2, 12.2, 17.7, 12.7),
    ("f16", 22, 17, 151, 151, 16.1, 14.5, 18.5, 16.1),
    ("u8", 43, 17, 151, 151, 27.5, 18.2, 30.8, 15.2),
    ("f16", 43, 17, 151, 151, 28.7, 22.7, 32.4, 24.9),
    ("u8", 1, 75, 59, 59, 2.6, 4.5, 2.7, 5.0),
    ("f16", 1, 75, 59, 59, 2.7, 4.3, 2.7, 5.0),
    ("u8", 1, 75, 83, 83, 2.7, 4.6, 2.9, 5.1),
    ("f16", 1, 75, 83, 83, 2.7, 4.3, 3.0, 5.1),
    ("u8", 1, 75, 119, 119, 3.3, 4.7, 3.5, 5.3),
    ("f16", 1, 75, 119, 119, 4.2, 5.3, 4.3, 6.0),
    ("u8", 1, 75, 167, 167, 5.0, 5.7, 6.1, 5.8),
    ("f16", 1, 75, 167, 167, 5.3, 7.0, 6.5, 8.0),
    ("u8", 2, 75, 151, 151, 7.6, 7.1, 8.1, 7.3),
    ("f16", 2, 75, 151, 151, 8.5, 8.7, 8.7, 8.9),
    ("u8", 5, 75, 151, 151, 13.9, 10.4, 14.3, 13.2),
    ("f16", 5, 75, 151, 151, 16.1, 13.7, 16.2, 14.3),
    ("u8", 10, 75, 151, 151, 24.9, 15.9, 24.7, 15.3),
    ("f16", 10, 75, 151, 151, 35.5, 23.0, 37.1, 26.3),
    ("u8", 1, 155, 41, 41, 2.7, 4.7, 2.7, 4.7),
    ("f16", 1, 155, 41, 41, 2.7, 5.0, 2.7, 4.9),
    ("u8", 1, 155, 59, 59, 2.9, 4.8, 2.9, 4.8),
    ("f16", 1, 155, 59, 59, 2.9, 5.1, 3.0, 5.1),
    ("u8", 1, 155, 83, 83, 3.0, 4.9, 3.6, 5.0),
    ("f16", 1, 155, 83, 83, 3.6, 5.8, 4.2, 6.2),
    ("u8", 1, 155, 117, 117, 5.8, 6.1, 6.3, 6.2),
    ("f16", 1, 155, 117, 117, 6.5, 8.2, 6.6, 8.2),
    ("u8", 1, 155, 165, 165, 8.7, 8.3, 8.8, 8.0),
    ("f16", 1, 155, 165, 165, 9.7, 10.5, 9.7, 10.2),
    ("u8", 2, 155, 151, 151, 11.6, 10.0, 11.8, 9.2),
    ("f16", 2, 155, 151, 151, 13.2, 13.4, 13.3, 13.6),
    ("u8", 5, 155, 151, 151, 23.7, 15.1, 23.9, 14.5),
    ("f16", 5, 155, 151, 151, 36.4, 26.9, 35.1, 27.1),
]


@pytest.mark.parametrize("row", RELAYOUT, ids=lambda r: "x".join(str(v) for v in r[:5]))
def test_relayout_takes_the_quicker_kernel(rules, row):
    dt, n, c, h, w, there32, there, back32, back = row
    for rows, cols, small, tile in ((c, h * w, there32, there), (h * w, c, back32, back)):
        chosen = tile if rules.transpose(SIZE[dt], n, rows, cols, CUS) else small
        assert chosen <= NEAR * min(small, tile)


# (operation, type, N, C, H, W, lanes, us with a thread per element -- rows of whole dwords: dword by dword --, us through tiles)
PACK = [
    ("pack", "u8", 1, 75, 14, 14, 4, 3.6, 3.8),
    ("pack", "u8", 1, 75, 14, 14, 32, 4.1, 3.9),
    ("pack", "f16", 1, 75, 14, 14, 16, 4.1, 4.0),
    ("pack", "u8", 1, 75, 19, 19, 4, 3.2, 4.0),
    ("pack", "u8", 1, 75, 19, 19, 32, 3.2, 4.1),
    ("unpack", "u8", 1, 75, 19, 19, 16, 2.6, 3.3),
    ("pack", "f16", 1, 75, 19, 19, 4, 3.2, 4.2),
    ("pack", "f16", 1, 75, 19, 19, 32, 3.2, 4.2),
    ("unpack", "f16", 1, 75, 19, 19, 32, 2.7, 3.5),
    ("pack", "f32", 1, 75, 19, 19, 16, 5.5, 4.2),
    ("pack", "u8", 1, 75, 38, 38, 16, 5.3, 4.1),
    ("pack", "u8", 1, 75, 51, 51, 4, 4.3, 4.2),
    ("pack", "u8", 1, 75, 51, 51, 32, 4.5, 4.2),
    ("unpack", "u8", 1, 75, 51, 51, 32, 3.0, 3.4),
    ("pack", "f16", 1, 75, 51, 51, 16, 4.4, 4.3),
    ("unpack", "f16", 1, 75, 51, 51, 16, 3.0, 3.5),
    ("pack", "f32", 1, 75, 51, 51, 4, 4.3, 4.4),
    ("pack", "u8", 1, 75, 75, 75, 4, 5.8, 4.3),
    ("unpack", "u8", 1, 75, 75, 75, 16, 3.4, 3.5),
    ("pack", "f16", 1, 75, 75, 75, 4, 5.8, 4.4),
    ("unpack", "f16", 1, 75, 75, 75, 4, 3.4, 4.8),
    ("unpack", "f16", 1, 75, 75, 75, 32, 4.0, 3.6),
    ("pack", "f32", 1, 75, 75, 75, 16, 6.4, 4.7),
    ("pack", "u8", 1, 75, 150, 150, 4, 4.6, 4.8),
    ("pack", "u8", 1, 75, 150, 150, 32, 6.2, 4.8),
    ("pack", "f16", 1, 75, 150, 150, 16, 6.7, 6.0),
    ("pack", "f32", 2, 75, 201, 201, 4, 14.6, 16.5),
    ("pack", "f32", 2, 75, 201, 201, 32, 17.5, 17.6),
    ("pack", "f32", 4, 75, 201, 201, 16, 28.9, 30.8),
    ("pack", "u8", 8, 75, 150, 150, 4, 11.1, 12.4),
    ("pack", "u8", 8, 75, 150, 150, 32, 11.4, 11.6),
    ("pack", "f16", 8, 75, 150, 150, 16, 16.0, 15.9),
    ("pack", "f32", 8, 75, 151, 151, 4, 30.6, 36.5),
    ("pack", "f32", 8, 75, 151, 151, 32, 32.9, 34.3),
    ("pack", "u8", 1, 155, 14, 14, 32, 4.1, 4.0),
    ("pack", "f16", 1, 155, 14, 14, 32, 5.7, 4.1),
    ("pack", "u8", 1, 155, 19, 19, 32, 3.3, 4.1),
    ("pack", "f16", 1, 155, 19, 19, 4, 3.3, 4.2),
    ("unpack", "f16", 1, 155, 19, 19, 32, 2.8, 3.5),
    ("pack", "u8", 1, 155, 38, 38, 4, 4.2, 4.1),
    ("pack", "f16", 1, 155, 38, 38, 4, 4.1, 4.2),
    ("pack", "u8", 1, 155, 51, 51, 32, 5.7, 4.2),
    ("unpack", "u8", 1, 155, 51, 51, 32, 3.4, 3.5),
    ("pack", "f16", 1, 155, 51, 51, 32, 6.1, 4.3),
    ("unpack", "f16", 1, 155, 51, 51, 32, 3.5, 3.6),
    ("pack", "f32", 1, 155, 51, 51, 32, 6.3, 4.5),
    ("unpack", "u8", 1, 155, 75, 75, 32, 4.9, 3.6),
    ("pack", "f32", 1, 155, 75, 75, 4, 5.2, 6.1),
    ("pack", "u8", 1, 155, 150, 150, 4, 5.2, 6.4),
    ("pack", "f16", 1, 155, 150, 150, 4, 7.3, 8.0),
    ("pack", "f32", 2, 155, 201, 201, 4, 28.3, 34.1),
    ("pack", "f32", 4, 155, 201, 201, 4, 49.2, 58.7),
    ("pack", "u8", 8, 155, 150, 150, 4, 16.6, 18.7),
    ("pack", "f16", 8, 155, 150, 150, 4, 27.5, 35.7),
    ("pack", "f32", 8, 155, 151, 151, 4, 53.4, 63.2),
    ("pack", "u8", 16, 3, 201, 201, 32, 153.9, 10.1),
    ("unpack", "u8", 16, 3, 201, 201, 32, 13.2, 7.7),
    ("unpack", "u8", 1, 75, 19, 19, 32, 2.7, 3.4),
    ("pack", "f32", 1, 75, 19, 19, 32, 6.1, 4.2),
    ("pack", "u8", 8, 155, 151, 151, 32, 204.3, 15.7),
    ("unpack", "u8", 8, 155, 151, 151, 32, 83.9, 12.5),
    ("pack", "f16", 8, 155, 151, 151, 32, 211.8, 31.8),
    ("unpack", "f16", 8, 155, 151, 151, 32, 128.8, 30.6),
    ("pack", "f32", 8, 155, 151, 151, 32, 54.0, 56.2),
]


@pytest.mark.parametrize("row", PACK, ids=lambda r: "-".join(str(v) for v in r[:7]))
def test_pack_takes_the_quicker_kernel(rules, row):
    op, dt, n, c, h, w, lanes, other, tiles = row
    es, plain, packed = SIZE[dt], n * c * h * w, n * -(-c // lanes) * lanes * h * w
    if h * w * es % 4:
        taken = rules.tile(es, lanes, plain, packed, op == "pack", CUS)
    else:
        taken = rules.pieces(lanes, h * w * es, plain * es)
    assert (tiles if taken else other) <= NEAR * min(other, tiles)
