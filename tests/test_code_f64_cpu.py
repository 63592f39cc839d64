"""``mdq_code_f64`` (csrc/mdq_math.h, the requant of 17..32-bit codes) compiled for the CPU against the
reference's own arithmetic, an IEEE double division and round half away, clamped, NaN as 0
(stquant_kernel.cu:366-381): exact ties and their neighbours, quotients next to 1/2 and to powers of
two, quotients beyond the range, zeros, subnormals, infinite and NaN divisors.  The two kinds of pairs
that it is not for, and that no block of a step has, are labelled as such."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stream-mm2026_amd", "csrc")

SRC = r"""
#include "mdq_math.h"
extern "C" void codes(const float *u, const float *d, uint32_t *out, long n, double lim)
{
    for (long i = 0; i < n; ++i) out[i] = mdq::mdq_code_f64(u[i], d[i], 1.0 / (double)d[i], lim);
}
"""


@pytest.fixture(scope="module")
def codes(tmp_path_factory):
    d = tmp_path_factory.mktemp("code_f64")
    (d / "c.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC,
                    "-o", str(d / "c.so"), str(d / "c.cpp")], check=True)
    fn = ctypes.CDLL(str(d / "c.so")).codes
    fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_long, ctypes.c_double]

    def run(u, dd, lim):
        u, dd = np.ascontiguousarray(u, np.float32), np.ascontiguousarray(dd, np.float32)
        out = np.empty(u.size, np.uint32)
        fn(u.ctypes.data, dd.ctypes.data, out.ctypes.data, u.size, float(lim))
        return out

    return run


def reference(u, d, lim):
    with np.errstate(all="ignore"):
        q = u.astype(np.float64) / d.astype(np.float64)
        t = np.trunc(q)
        k = np.where(np.isinf(q), q, t + (np.abs(q - t) >= 0.5))
    return np.clip(np.where(np.isnan(q), 0.0, k), 0.0, lim).astype(np.uint32)


@pytest.mark.parametrize("bits", [17, 24, 31, 32])
def test_equals_the_fp64_division_and_round(codes, bits):
    rng = np.random.default_rng(bits)
    n = 400_000
    for lim in (2.0 ** bits - 1, 2.0 ** (bits - 1) - 1, 2.0 ** (bits - 1)):
        d = np.exp(rng.uniform(np.log(1e-12), 40, n)).astype(np.float32)
        k = np.floor(np.exp(rng.uniform(0, np.log(2.0 ** bits), n)))
        u = ((k + rng.choice([0.0, 0.5, 0.25, -0.5], n)) * d.astype(np.float64)).astype(np.float32)
        for step in (0, 1, -1):                       # the product's float and its neighbours
            v = u if step == 0 else np.nextafter(u, np.float32(np.inf * step), dtype=np.float32)
            v = np.maximum(v, np.float32(0))
            np.testing.assert_array_equal(codes(v, d, lim), reference(v, d, lim))
        p2 = (2.0 ** rng.integers(-40, 40, n)).astype(np.float32)      # exact quotients: ties of every size
        for w in (k + 0.5, 2.0 ** rng.integers(0, bits, n) - 0.5):
            v = (w.astype(np.float32).astype(np.float64) * p2).astype(np.float32)
            np.testing.assert_array_equal(codes(v, p2, lim), reference(v, p2, lim))
        h = (d.astype(np.float64) * 0.5).astype(np.float32)            # u / d next to 1/2
        for v in (h, np.nextafter(h, np.float32(0)), np.nextafter(h, np.float32(np.inf))):
            np.testing.assert_array_equal(codes(v, d, lim), reference(v, d, lim))


def test_edges(codes):
    f = np.float32
    fmax, tiny, inf, nan = np.finfo(f).max, f(1e-45), f(np.inf), f(np.nan)
    u = np.array([0, 0, tiny, tiny, fmax, fmax, fmax, inf, inf, 1, nan, 1, nan, 3, fmax], f)
    d = np.array([1e-12, inf, 1e-12, fmax, 1e-12, fmax, 2 * tiny, inf, nan, inf, 1, nan, nan, 2, 1], f)
    for lim in (2.0 ** 32 - 1, 2.0 ** 31, 2.0 ** 17 - 1):
        np.testing.assert_array_equal(codes(u, d, lim), reference(u, d, lim))


def test_pairs_that_no_block_has(codes):
    """An infinite u over a finite d, and u > 0 over d = 0: 0, where the division would clamp to lim.  The
    divisor of a block is infinite or NaN where an element is, and at least 1e-12 over the range."""
    u, d = np.array([np.inf, 1.0], np.float32), np.array([1.0, 0.0], np.float32)
    assert codes(u, d, 2.0 ** 31).tolist() == [0, 0]
    assert reference(u, d, 2.0 ** 31).tolist() == [2 ** 31, 2 ** 31]
