"""Arithmetic of the kernels that a host program can evaluate: the headers' own functions in a host build."""
import ctypes as C
import os
import subprocess
from pathlib import Path

import numpy as np
import pytest

from pcaone_amd import build

SOURCE = r'''
#include "small_la.hpp"
using namespace pcaone;
extern "C" {
void places(const double* x, int stride, int n, int* out) {
  for (int i = 0; i < n; ++i) out[i] = place_descending(x, stride, n, i);
}
void divisions(const double* x, const double* d, int n, double* out) {
  for (int i = 0; i < n; ++i) out[i] = quotient_any(x[i], d[i], 1.0 / d[i]);
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
