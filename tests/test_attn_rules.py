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
    (128, 16, 15583, 32.1, 21.7), (128, 8, 12668, 18.4, 20.0), (128, 1616, 64, 8.5, 10.4), (128, 8192, 16, 28.9, 38.1), (128, 4096, 112, 17.9, 19.1),
    (128, 260, 984, 22.4, 26.2), (128, 272, 711, 15.5, 17.5), (128, 288, 670, 16.1, 18.6), (128, 308, 690, 20.7, 19.0), (128, 332, 606, 19.5, 17.2), (128, 436, 622, 24.2, 20.1),
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


RUNS = [256, 384, 512, 768, 1024, 1536, 2048]
# sequences, kv heads of 128, tokens together, tokens of the longest, us with splits of RUNS tokens (evenly from 0.9 of the longest to the
# longest, from a half of it, from an eighth, or one long one and the rest 400), in caches of two to fifty times the longest
LENGTHS = [
    (4, 8, 1140, 300, 8.5, 7.4, 7.4, 7.3, 7.4, 7.3, 7.4),
    (4, 8, 3800, 1000, 9.0, 10.0, 11.0, 13.2, 13.6, 13.6, 13.6),
    (4, 8, 12920, 3400, 16.4, 18.9, 15.1, 17.4, 19.4, 24.0, 29.3),
    (4, 8, 30400, 8000, 30.7, 30.6, 28.7, 32.8, 26.9, 28.3, 32.7),
    (4, 8, 49152, 16384, 50.2, 50.0, 45.7, 46.7, 43.6, 53.1, 39.3),
    (4, 8, 65536, 16384, 57.9, 57.7, 54.4, 54.2, 51.4, 59.5, 49.7),
    (4, 8, 36864, 16384, 44.1, 44.1, 40.0, 42.3, 38.0, 47.4, 34.0),
    (32, 1, 30400, 1000, 8.8, 9.8, 10.7, 12.8, 13.2, 13.1, 13.2),
    (32, 1, 103360, 3400, 17.2, 19.3, 16.0, 18.7, 20.9, 24.4, 29.3),
    (16, 8, 15200, 1000, 17.8, 18.3, 17.0, 19.2, 19.5, 19.7, 19.7),
    (16, 8, 30400, 2000, 29.7, 30.1, 28.5, 29.9, 27.9, 31.9, 33.5),
    (16, 8, 65536, 4096, 56.5, 55.9, 53.6, 54.7, 52.1, 56.1, 51.4),
    (16, 8, 10096, 4096, 18.3, 21.9, 25.4, 33.3, 30.1, 35.2, 29.2),
    (2, 8, 1900, 1000, 8.7, 9.6, 10.5, 12.7, 13.1, 13.1, 13.1),
    (2, 8, 6460, 3400, 12.0, 12.0, 12.2, 14.3, 16.6, 21.1, 25.9),
    (2, 8, 15200, 8000, 20.8, 21.2, 18.7, 19.4, 22.2, 26.2, 29.9),
    (10, 8, 9500, 1000, 13.7, 12.5, 13.9, 15.9, 16.3, 16.2, 16.2),
    (10, 8, 19000, 2000, 21.7, 21.1, 22.8, 20.3, 21.4, 27.0, 29.7),
    (10, 8, 6600, 3000, 14.4, 15.0, 16.4, 14.3, 16.7, 21.5, 26.5),
    (64, 4, 60800, 1000, 25.1, 24.7, 24.8, 24.8, 22.7, 22.7, 22.7),
    (64, 4, 121600, 2000, 51.0, 49.4, 48.0, 47.3, 47.3, 47.1, 44.5),
    (40, 1, 76000, 2000, 14.2, 12.8, 13.8, 15.8, 17.8, 23.1, 26.0),
]


@pytest.fixture(scope="module")
def run_by_lengths(tmp_path_factory):
    d = tmp_path_factory.mktemp("lengths")
    (d / "r.cpp").write_text("""#include "attn_rules.hpp"
extern "C" int run_by_lengths(long batch, long kv_heads, unsigned longest, unsigned total, long most) {
    return nnhip::attn_run(nnhip::attn_run_rule(batch, kv_heads, 256, most), longest, total);
}
extern "C" long most_splits(long pairs, long capacity, int run) { return nnhip::attn_most_splits(pairs, capacity, run); }
""")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "r.cpp"), "-o", str(d / "r.so")])
    lib = C.CDLL(str(d / "r.so"))
    lib.run_by_lengths.argtypes = [C.c_long, C.c_long, C.c_uint, C.c_uint, C.c_long]
    lib.most_splits.argtypes, lib.most_splits.restype = [C.c_long, C.c_long, C.c_int], C.c_long
    return lib


@pytest.mark.parametrize("row", LENGTHS, ids=lambda r: "%dx%d-%d-%d" % (r[0], r[1], r[3], r[2]))
def test_splits_follow_the_lengths_not_the_capacity(run_by_lengths, row):
    """(A run between two measured ones is held to the slower of them.)"""
    run = run_by_lengths.run_by_lengths(row[0], row[1], row[3], row[2], 1024)
    near = [t for r, t in zip(RUNS, row[4:]) if r == run] or [t for r, t, n in zip(RUNS, row[4:], RUNS[1:] + [0]) if r < run < n or r == min(x for x in RUNS if x > run)]
    assert max(near) <= 1.125 * min(row[4:]), (run, near)


def test_every_split_of_a_sequence_has_its_blocks(run_by_lengths, choose_run):
    """Whatever the lengths: whole steps, no more splits than the launch has blocks for, and the capacity's run for full contexts."""
    for kv_heads in (1, 2, 8, 30):
        for batch in (1, 2, 3, 16, 33, 64, 65, 200, 256):
            pairs = batch * kv_heads
            if not 16 <= pairs <= 256: continue
            for capacity in (400, 1024, 1040, 3000, 4096, 16384, 131072, 1 << 20, 1 << 21):
                run = choose_run(128, pairs, capacity, 256)
                if run == 0: continue
                least = -(-capacity // run)
                most = run_by_lengths.most_splits(pairs, capacity, run)
                assert least <= most <= max(least, 1024)
                assert run_by_lengths.run_by_lengths(batch, kv_heads, capacity, capacity * batch, most) == run
                for room in {least, most}:                       # (as many as the scratch there is has room for)
                    for longest in {1, 127, 128, 129, 383, 384, 385, 511, 513, 1023, 1025, 2047, 2049, capacity // 2 + 1, capacity - 1, capacity}:
                        if longest > capacity: continue
                        for total in {longest, longest + (batch - 1) * (longest // 9), longest * batch}:
                            r = run_by_lengths.run_by_lengths(batch, kv_heads, longest, total, room)
                            assert r > 0 and r % 128 == 0 and r * room >= longest, (batch, kv_heads, capacity, longest, total, r)


@pytest.mark.parametrize("batch,kv_heads,longest", [(16, 1, 300), (24, 1, 439), (13, 4, 468), (52, 2, 487), (4, 8, 512), (200, 1, 512)])
def test_short_contexts_in_a_large_cache_are_one_split(run_by_lengths, batch, kv_heads, longest):
    """(us with two splits / one: 24 x 1 of 439 tokens 10.9 / 8.9, 13 x 4 of 468 9.2 / 8.4, 52 x 2 of 487 9.2 / 8.5)"""
    for total in (longest * batch, longest + (batch - 1) * (longest // 5)):
        assert run_by_lengths.run_by_lengths(batch, kv_heads, longest, total, 64) >= longest
    assert run_by_lengths.run_by_lengths(batch, kv_heads, 640, 640 * batch, 64) < 640 or batch * kv_heads > 128
