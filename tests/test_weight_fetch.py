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
