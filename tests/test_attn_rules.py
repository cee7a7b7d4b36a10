"""How paged attention splits a context over blocks, held against measured times (us on the device, 256 compute units; contexts
between filled and a half): the choice is never more than an eighth slower than the best of the block shapes.  The rule is host
arithmetic (csrc/attn_rules.hpp), compiled here for the CPU."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nncase_amd", "csrc")
SHAPES = [(2, 4), (4, 4), (2, 8), (4, 8)]   # tiles per wave, waves


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text("""#include "attn_rules.hpp"
extern "C" int choose(int head_dim, long pairs, long tokens, int cus) {
    const nnhip::AttnBlock b = nnhip::choose_attn_block(head_dim, pairs, tokens, cus);
    return b.tiles * 16 + b.waves;
}
""")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "r.cpp"), "-o", str(d / "r.so")])
    fn = C.CDLL(str(d / "r.so")).choose
    fn.argtypes = [C.c_int, C.c_long, C.c_long, C.c_int]
    return lambda *a: divmod(fn(*a), 16)


# head_dim, pairs of sequence and kv head, capacity in tokens, us as 2 x 4, 4 x 4, 2 x 8, 4 x 8 (tiles x waves)
MEASURED = [
    (64, 2, 112, 4.1, 4.4, 4.2, 4.5),
    (64, 2, 256, 5.9, 5.1, 5.0, 5.2),
    (64, 2, 704, 6.3, 6.8, 6.9, 8.2),
    (64, 2, 2064, 8.1, 8.0, 8.2, 8.8),
    (64, 2, 3504, 8.1, 8.2, 8.3, 9.0),
    (64, 2, 16000, 18.1, 12.5, 11.2, 10.8),
    (64, 4, 208, 5.9, 5.0, 4.8, 5.1),
    (64, 8, 112, 4.2, 4.4, 4.3, 4.5),
    (64, 8, 512, 6.3, 7.0, 7.3, 6.7),
    (64, 12, 2064, 8.3, 8.0, 8.0, 8.8),
    (64, 12, 4096, 10.0, 8.8, 8.8, 9.2),
    (64, 12, 10000, 17.0, 12.5, 12.6, 11.1),
    (64, 24, 2064, 10.6, 9.2, 9.3, 9.5),
    (64, 24, 4112, 11.2, 9.5, 9.5, 9.5),
    (64, 32, 208, 6.4, 5.2, 5.0, 5.3),
    (64, 48, 112, 3.9, 4.2, 4.2, 4.5),
    (64, 48, 8192, 21.0, 16.9, 17.6, 18.9),
    (64, 64, 8192, 27.0, 21.7, 23.8, 22.4),
    (64, 96, 112, 4.2, 4.5, 4.4, 4.7),
    (64, 96, 704, 8.3, 8.5, 8.8, 9.0),
    (64, 128, 3504, 19.9, 17.7, 19.8, 20.4),
    (64, 144, 144, 6.1, 4.6, 4.5, 4.9),
    (64, 288, 2048, 19.3, 19.5, 20.7, 22.5),
    (128, 4, 112, 5.4, 5.9, 5.7, 6.2),
    (128, 4, 704, 8.4, 9.5, 9.0, 12.0),
    (128, 8, 208, 6.7, 6.9, 6.4, 7.3),
    (128, 8, 3008, 10.3, 10.5, 10.7, 12.6),
    (128, 8, 4112, 16.1, 14.0, 12.1, 14.0),
    (128, 8, 8000, 17.5, 14.0, 13.6, 14.6),
    (128, 16, 112, 5.1, 5.6, 5.4, 6.0),
    (128, 16, 2064, 13.9, 12.7, 11.4, 13.2),
    (128, 32, 144, 7.0, 6.3, 5.8, 6.6),
    (128, 32, 304, 7.2, 8.9, 8.9, 8.2),
    (128, 32, 4112, 17.5, 15.1, 13.9, 13.4),
    (128, 32, 8000, 35.6, 29.8, 28.4, 30.2),
    (128, 64, 6000, 24.4, 21.8, 23.5, 25.4),
    (128, 64, 10000, 34.8, 32.3, 37.4, 44.4),
    (128, 128, 2048, 19.6, 18.1, 20.9, 23.9),
    (128, 256, 208, 9.8, 8.1, 7.8, 8.4),
    (128, 400, 112, 7.6, 8.0, 8.4, 11.8),
]


@pytest.mark.parametrize("row", MEASURED, ids=lambda r: "%d-%d-%d" % r[:3])
def test_context_is_split_into_the_quicker_blocks(choose, row):
    assert row[3 + SHAPES.index(choose(row[0], row[1], row[2], 256))] <= 1.125 * min(row[3:])


def test_every_choice_is_a_kernel_that_is_built(choose):
    for d in (64, 128):
        for pairs in (1, 3, 8, 30, 64, 200, 256, 257, 1000, 100000):
            for tokens in list(range(1, 1200, 37)) + [2048, 3200, 4096, 4112, 6500, 9999, 10000, 16384, 131072, 1 << 20]:
                assert choose(d, pairs, tokens, 256) in SHAPES


# head_dim, pairs, capacity in tokens, us of the block chosen above, us with the split gone through in steps
STEPS = [
    (64, 12, 433, 6.2, 6.4), (64, 24, 265, 5.8, 5.3), (64, 60, 459, 6.6, 6.2), (64, 240, 384, 7.8, 5.9), (64, 84, 4759, 16.4, 17.9),
    (64, 144, 3041, 16.7, 18.2), (64, 132, 14756, 50.7, 52.1), (128, 64, 1205, 12.1, 13.0), (128, 8, 4387, 12.3, 14.0), (128, 4, 993, 8.6, 9.3),
    (128, 36, 6028, 22.3, 17.9), (128, 104, 9746, 106.9, 79.6), (128, 256, 490, 13.0, 10.2), (128, 624, 280, 21.6, 19.0), (128, 656, 4073, 266.7, 229.1),
    (128, 16, 15583, 32.1, 21.7), (128, 8, 12668, 18.4, 20.0),
]


@pytest.fixture(scope="module")
def choose_run(tmp_path_factory):
    d = tmp_path_factory.mktemp("run")
    (d / "r.cpp").write_text("""#include "attn_rules.hpp"
extern "C" int choose_run(int head_dim, long pairs, long tokens, int cus) { return nnhip::choose_attn_run(head_dim, pairs, tokens, cus); }
""")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "r.cpp"), "-o", str(d / "r.so")])
    fn = C.CDLL(str(d / "r.so")).choose_run
    fn.argtypes = [C.c_int, C.c_long, C.c_long, C.c_int]
    return fn


@pytest.mark.parametrize("row", STEPS, ids=lambda r: "%d-%d-%d" % r[:3])
def test_steps_are_taken_where_they_are_quicker(choose_run, row):
    assert (choose_run(row[0], row[1], row[2], 256) > 0) == (row[4] < row[3])


def test_runs_are_whole_steps(choose_run):
    for d in (64, 128):
        for pairs in (1, 16, 24, 30, 64, 200, 256, 257, 1000, 100000, 1 << 30):
            for tokens in list(range(1, 1200, 37)) + [2048, 4112, 9999, 131072, 1 << 20, (1 << 31) - 1]:
                run = choose_run(d, pairs, tokens, 256)
                assert run % 128 == 0 and 0 <= run <= 2048
                assert run == 0 or d == 128 or run >= tokens      # (64-wide heads: one split alone)
