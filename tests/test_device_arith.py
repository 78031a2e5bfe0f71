"""Arithmetic of the kernels that a host program can evaluate: the headers' own functions in a host build."""
import ctypes as C
import os
import subprocess
from pathlib import Path

import numpy as np
import pytest

from pcaone_amd import build

SOURCE = r'''
#include "bf16.hpp"
#include "small_la.hpp"
using namespace pcaone;
extern "C" {
void places(const double* x, int stride, int n, int* out) {
  for (int i = 0; i < n; ++i) out[i] = place_descending(x, stride, n, i);
}
void divisions(const double* x, const double* d, int n, double* out) {
  for (int i = 0; i < n; ++i) out[i] = quotient_any(x[i], d[i], 1.0 / d[i]);
}
void roots(const double* d, const double* y0, int n, double* r, double* inv) {
  for (int i = 0; i < n; ++i) refine_root(d[i], y0[i], r[i], inv[i]);
}
void e4m3(const double* x, int n, unsigned char* bits, double* value) {
  for (int i = 0; i < n; ++i) bits[i] = e4m3_bits(x[i], &value[i]);
}
}
'''


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("arith")
    (d / "arith.cpp").write_text(SOURCE)
    subprocess.run([build.HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-std=c++20", "-fPIC", "-shared",
                    "-march=x86-64-v3", "-ffp-contract=off", "-Wno-unused-function", f"-I{build.CSRC}",
                    str(d / "arith.cpp"), "-o", str(d / "arith.so")], check=True, timeout=300)
    return C.CDLL(str(d / "arith.so"))


def dptr(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


@pytest.mark.parametrize("values", [[3.0, 1.0, 2.0], [0.0, -0.0, 0.0, 1.0], [np.nan] * 5, [1.0, np.nan, 2.0, np.nan],
                                    [np.inf, np.nan, -np.inf, np.inf, 0.0], [5.0], [np.nan]])
def test_descending_places_are_a_permutation(host, values):
    """The batched eigen-solver scatters its indexes to these places and reads columns by them: every place is
    taken once whatever the values, numbers in descending order and NaNs after them."""
    n, stride = len(values), 3
    x = np.full(n * stride, 7.0)
    x[::stride] = values
    out = np.full(n, -1, np.int32)
    host.places(dptr(x), stride, n, out.ctypes.data_as(C.POINTER(C.c_int)))
    assert sorted(out) == list(range(n))
    ordered = np.empty(n)
    ordered[out] = values
    numbers = ordered[~np.isnan(ordered)]
    assert not np.isnan(ordered[:len(numbers)]).any()
    assert np.all(numbers[:-1] >= numbers[1:])


def divisions(host, x, d):
    x, d = np.ascontiguousarray(x, dtype=np.float64), np.ascontiguousarray(d, dtype=np.float64)
    out = np.empty_like(x)
    host.divisions(dptr(x), dptr(d), len(x), dptr(out))
    return out


def test_divisions_round_as_the_quotient(host):
    """Random significands and exponents (and quotients next to ties and to 1): the very bits of x / d."""
    rng = np.random.default_rng(1)
    n = 200000
    x = np.ldexp(1 + rng.random(n), rng.integers(-400, 400, n)) * rng.choice([-1, 1], n)
    d = np.ldexp(1 + rng.random(n), rng.integers(-400, 400, n))
    near = 1 + rng.integers(0, 64, n) * 2.0**-52
    for a, b in ((x, d), (d * near, d), (near, 1 + rng.integers(0, 64, n) * 2.0**-52), (x, np.sqrt(d))):
        np.testing.assert_array_equal(divisions(host, a, b), a / b)


def test_divisions_of_infinities_and_zeros(host):
    """Dividends that are zero, infinite, NaN or the smallest that the residual allows, and overflow."""
    x = np.array([0.0, -0.0, 1.0, -3.0, np.inf, -np.inf, np.nan, 1e308, -1.7e308, 2.0**-960, -3 * 2.0**-959])
    x, d = (a.ravel() for a in np.meshgrid(x, [1.0, 3.0, 1.4142135e9, 0.125, 1e-4]))
    with np.errstate(all="ignore"):
        ref = x / d
    np.testing.assert_array_equal(divisions(host, x, d), ref)


def test_roots_round_as_sqrt_and_its_reciprocal(host):
    """Random significands, squares and their neighbours, estimates off by up to 2^-23 both ways: the very bits of
    sqrt(d) and of 1 / sqrt(d)."""
    rng = np.random.default_rng(2)
    n = 300000
    d = np.ldexp(1 + rng.random(n), rng.integers(-300, 300, n))
    s = 1 + rng.integers(0, 2**26, n) * 2.0**-26
    square = s * s
    for x in (d, square, np.nextafter(square, 0), np.nextafter(square, 9)):
        y0 = 1 / np.sqrt(x) * (1 + rng.uniform(-1, 1, n) * 2.0**-23)
        r, inv = np.empty(n), np.empty(n)
        host.roots(dptr(x), dptr(y0), n, dptr(r), dptr(inv))
        np.testing.assert_array_equal(r, np.sqrt(x))
        plain = np.frexp(r)[0] != 1 - 2.0**-53  # r of all ones: the stated exception
        np.testing.assert_array_equal(inv[plain], (1 / r)[plain])


def test_e4m3_is_the_nearest_code(host):
    """Every non-negative code's value, the ties between neighbours (to the even code) and the FP64 numbers beside
    them, subnormal codes among them, the largest value and all beyond it; both signs."""
    codes = np.arange(0x7F)  # 0x7F is NaN
    e, f = codes >> 3, codes & 7
    table = np.where(e == 0, np.ldexp(f / 8.0, -6), np.ldexp(1 + f / 8.0, e - 7))
    mid = (table[1:] + table[:-1]) / 2
    x = np.concatenate([table, mid, np.nextafter(mid, 0), np.nextafter(mid, 1e9), np.nextafter(table, 1e9),
                        [464.0, 480.0, 1e6, 1e300, np.inf, 5e-324, 1e-310, 2.0**-11]])
    x = np.concatenate([x, -x, [np.nan]])
    bits, value = np.zeros(len(x), np.uint8), np.empty(len(x))
    host.e4m3(dptr(x), len(x), bits.ctypes.data_as(C.POINTER(C.c_ubyte)), dptr(value))
    for v, b, got in zip(x, bits, value):
        gap = np.abs(table - min(abs(v), 448.0)) if v == v else table
        near = np.flatnonzero(gap == gap.min())
        code = int(near[0]) if len(near) == 1 or near[0] % 2 == 0 else int(near[1])
        assert b == (code | (0x80 if v < 0 and code else 0)), (v, hex(b), hex(code))
        assert got == np.copysign(table[code], v) or (v != v and got == 0)
