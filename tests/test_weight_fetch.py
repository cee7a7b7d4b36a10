"""Which fragments of packed weights an attention launch brings into the caches (csrc/weight_fetch.hpp): over the dies, every fragment
of every product once, on the die whose blocks read it, and never one outside the weights.  Host arithmetic, compiled here for the CPU."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nncase_amd", "csrc")
BASE = 1 << 32


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("fetch")
    (d / "f.cpp").write_text("""#include "weight_fetch.hpp"
using namespace nnhip;
static WeightFetches make(const unsigned *p, int n) {
    WeightFetches s = {};
    for (s.count = 0; s.count < n; s.count++, p += 4) s.f[s.count] = {(const void *)((size_t)(s.count + 1) << 32), p[0], p[1], p[2], p[3]};
    return s;
}
extern "C" unsigned fragments(const unsigned *p, int i, unsigned x) { return fetch_fragments(make(p, i + 1).f[i], x); }
extern "C" size_t address(const unsigned *p, int n, unsigned x, unsigned u) { return (size_t)fetch_address(make(p, n), x, u); }
""")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "f.cpp"), "-o", str(d / "f.so")])
    lib = C.CDLL(str(d / "f.so"))
    lib.address.restype = C.c_size_t
    return lib


# (blocks, k-steps, tiles between a block's two, tiles per block) of each product
@pytest.mark.parametrize("products", [
    [(56, 14, 56, 1), (304, 14, 304, 2), (56, 76, 56, 1), (36, 14, 2, 2)],     # the benchmark's decode layer, head_dim 64
    [(1, 1, 1, 1)], [(3, 2, 3, 2)], [(13, 5, 13, 1), (12, 1, 4, 2)], [(8, 3, 1, 2), (9, 7, 9, 2), (200, 3, 200, 1)],
])
def test_every_fragment_once_on_its_die(lib, products):
    flat = (C.c_uint * (4 * len(products)))(*[v for p in products for v in p])
    seen = [[0] * (blocks * per * steps) for blocks, steps, _, per in products]
    for x in range(8):
        total = sum(lib.fragments(flat, i, x) for i in range(len(products)))
        for u in range(total):
            at = lib.address(flat, len(products), x, u)
            i, position = at // BASE - 1, at % BASE // 1024
            blocks, steps, off, per = products[i]
            seen[i][position] += 1
            tile = position // steps
            block = tile // (2 * off) * off + tile % off if per == 2 else tile
            assert block < blocks and block % 8 == x
    assert all(v == 1 for s in seen for v in s)


# lanes, rows of a lane, longest context, us a decode step of 24 layers without and with the weights fetched (2 kv heads of 64)
FETCHED = [
    (1, 1, 700, 654.8, 602.1), (1, 1, 16000, 757.2, 726.6), (1, 8, 8192, 838.0, 827.3), (1, 16, 700, 769.9, 752.9), (1, 32, 700, 894.5, 886.2),
    (2, 4, 700, 752.6, 730.7), (2, 4, 4096, 823.0, 806.5), (2, 6, 1500, 815.2, 806.0), (2, 8, 700, 793.0, 790.4), (2, 8, 4096, 901.4, 890.3), (2, 8, 8192, 962.8, 997.5),
    (2, 10, 1500, 864.2, 877.3), (2, 12, 1500, 879.5, 901.2), (2, 16, 700, 869.2, 885.1), (2, 16, 2048, 909.0, 953.1), (2, 16, 4096, 1037.4, 1069.2),
    (2, 32, 1000, 1046.8, 1066.9), (2, 32, 2048, 1138.4, 1179.8), (4, 2, 700, 1515.8, 1469.9), (4, 4, 1500, 1630.0, 1592.0), (4, 8, 700, 1667.7, 1643.2),
    (4, 16, 2048, 1961.8, 1991.5),
]


@pytest.mark.parametrize("lanes,rows,tokens,without,fetched", FETCHED)
def test_weights_are_fetched_where_that_is_the_quicker(tmp_path_factory, lanes, rows, tokens, without, fetched):
    d = tmp_path_factory.getbasetemp() / "beside"
    if not (d / "r.so").exists():
        d.mkdir(exist_ok=True)
        (d / "r.cpp").write_text("""#include "weight_fetch.hpp"
extern "C" int beside(int lanes, int rows, long kv_bytes) { return nnhip::fetch_beside_lanes(lanes, rows, kv_bytes); }
""")
        subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "r.cpp"), "-o", str(d / "r.so")])
    fn = C.CDLL(str(d / "r.so")).beside
    fn.argtypes = [C.c_int, C.c_int, C.c_long]
    assert bool(fn(lanes, rows, rows * 2 * tokens * 64 * 4)) == (fetched < without)
