"""Host-side quantisation-parameter maths (nncase_amd.quant) against the reference's literal
expectations and against the oracle's independent restatement."""
import json
import os

import numpy as np

from nncase_amd import quant
from oracle import oracle as O

GOLD = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "reference_vectors.json")))
f32 = np.float32


def test_literals():
    for g in GOLD["K4_get_quant_param"] + [GOLD["K6_quant_param_of"]]:
        zp, sc = quant.get_quant_param(tuple(g["range"]), g["bits"], quant.QuantMode[g["mode"]])
        assert zp == g["zero_point"] and sc == f32(g["scale"])
    for g in GOLD["K5_fixup_range"]:
        assert quant.fixup_range(tuple(g["range"]), g["symmetric"]) == (f32(g["expected"][0]), f32(g["expected"][1]))


def test_matches_oracle_on_random_ranges():
    rng = np.random.default_rng(0)
    for _ in range(3000):
        lo, hi = np.sort(rng.standard_normal(2).astype(f32) * f32(10 ** rng.uniform(-4, 3)))
        for mode in quant.QuantMode:
            assert quant.get_quant_param((lo, hi), 8, mode) == O.get_quant_param(lo, hi, 8, int(mode))
        assert quant.fixup_range((lo, hi)) == O.fixup_range(lo, hi)
        assert quant.calib_fixup_range((lo, hi)) == O.calib_fixup_range(lo, hi)


def test_calibration_union_and_weight_quantisation():
    samples = [np.array([0.5, 2.0, np.inf], f32), np.array([-1.0, 1.0, np.nan], f32)]
    assert quant.calibrate_range(samples) == (f32(-1.0), f32(2.0))
    rng = np.random.default_rng(1)
    w = (rng.standard_normal((8, 4, 3, 3)) * 0.05).astype(f32)
    q, zp, sc = quant.quantize_weights(w)
    assert (zp, sc) == O.get_quant_param(w.min(), w.max())
    assert np.array_equal(q, O.quantize(w, sc, zp, O.U8))


def test_division_by_the_reciprocal_is_exact(tmp_path):
    """x * r corrected once by the residual is the nearest float of x / b wherever the quotient lies so near to the middle of two floats
    that the correction's own error (at most 1.5 * 2^-24 ulp) could matter: for a mantissa b, the a with a * 2^24 or a * 2^25 = r mod b
    and |r| up to 6, found by the inverse of the power of two.  Every 64th b here; all of them have been held once."""
    import subprocess
    (tmp_path / "d.c").write_text("""
#include <math.h>
#include <stdint.h>
static int64_t inverse(int64_t x, int64_t m) {
    int64_t a = x % m, b = m, u = 1, v = 0;
    while (b) { int64_t t = a / b, s = a - t * b; a = b; b = s; s = u - t * v; u = v; v = s; }
    return (u % m + m) % m;
}
long held(int64_t first, long *tried) {
    long bad = 0, n = 0;
    for (int64_t b = (1 << 23) + first; b < 1 << 24; b += 64) {
        const float fb = (float)b, y = 1.0f / fb;
        const int t = __builtin_ctzll(b);
        const int64_t odd = b >> t;
        if (odd == 1 || t > 2) continue; /* (r would have to be a multiple of 8) */
        for (int s = 24; s <= 25; s++)
            for (int r = -6; r <= 6; r++) {
                if (!r || (r & ((1 << t) - 1))) continue;
                int64_t two = 1;
                for (int i = 0; i < s - t; i++) two = two * 2 % odd;
                for (int64_t a = (int64_t)((__int128)inverse(two, odd) * ((r >> t) + odd) % odd); a < 1 << 24; a += odd) {
                    if (a < 1 << 23) continue;
                    const float fa = (float)a, q0 = fa * y, q = fmaf(fmaf(-fb, q0, fa), y, q0);
                    n++, bad += q != fa / fb;
                }
            }
    }
    *tried = n;
    return bad;
}
""")
    subprocess.check_call(["gcc", "-O2", "-mfma", "-ffp-contract=off", "-shared", "-fPIC", str(tmp_path / "d.c"), "-o", str(tmp_path / "d.so"), "-lm"])
    import ctypes
    fn = ctypes.CDLL(str(tmp_path / "d.so")).held
    fn.argtypes, fn.restype = [ctypes.c_int64, ctypes.POINTER(ctypes.c_long)], ctypes.c_long
    tried = ctypes.c_long()
    for first in (1, 2, 63):
        assert fn(first, ctypes.byref(tried)) == 0 and tried.value > 100000
