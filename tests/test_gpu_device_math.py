"""The device forms of gam_math.h (hardware seed, two Newton or Goldschmidt
steps) and gam_erfc.h, which the host builds of the CPU tests replace by
plain operations, against 40-digit values over the range of exponents.

Bounds on the relative error, u = 2^-53.  Reciprocal and square roots end in
one fused correction of a value good to a few u: its rounding, u, and the
square of what was left before: 1.01 u.  The reciprocal square root ends in
a Goldschmidt step of h alone, which keeps half the difference of the
roundings of g and h: u / 2 from x y, u from the first step, and u of its own
rounding: 2.5 u.  exp and erfc: 1e-15, as on the host (test_erfc.py).
"""
import ctypes as C
import os

import mpmath as mp
import numpy as np
import pytest

from mage_amd import build

pytestmark = pytest.mark.gpu
DP = C.POINTER(C.c_double)
U = 2.0 ** -53
RCP, SQRT_RSQRT, SQRT, EXP, ERFC = range(5)


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(build.MATH_LIB):
        build.build_math_test_lib()
    L = C.CDLL(build.MATH_LIB)
    L.dev_math.argtypes = [C.c_int, C.c_int, DP, DP, DP]
    return L


def _eval(L, fn, x):
    x = np.ascontiguousarray(x, dtype=np.float64)
    y, e = np.empty_like(x), np.empty_like(x)
    assert L.dev_math(fn, len(x), *[a.ctypes.data_as(DP) for a in (x, y, e)]) == 0
    return y, e


def _range(lo, hi, n=3000):
    """n values of random mantissa, exponents spread over [lo, hi], and the
    ends of a binade."""
    r = np.random.default_rng(5)
    x = (1 + r.random(n)) * 2.0 ** r.integers(lo, hi, n)
    return np.concatenate([x, 2.0 ** np.arange(lo, hi, 7.0), (2 - 2.0 ** -52) * 2.0 ** np.arange(lo, hi, 7.0)])


def _worst(x, y, f):
    mp.mp.dps = 40
    return max(float(abs(mp.mpf(float(b)) / f(mp.mpf(float(a))) - 1)) for a, b in zip(x, y))


def test_reciprocal(lib):
    x = _range(-1000, 1000)
    x[::2] *= -1               # the determinant of an edge's directions has either sign
    assert _worst(x, _eval(lib, RCP, x)[0], lambda v: 1 / v) <= 1.01 * U


def test_square_roots(lib):
    x = _range(-1000, 1000)
    s, r = _eval(lib, SQRT_RSQRT, x)
    assert _worst(x, s, mp.sqrt) <= 1.01 * U
    assert _worst(x, r, lambda v: 1 / mp.sqrt(v)) <= 2.5 * U
    x = _range(-929, 1000)     # above 1e-280
    assert _worst(x, _eval(lib, SQRT, x)[0], mp.sqrt) <= 1.01 * U
    y = _eval(lib, SQRT, np.array([0.0, 5e-324, 1e-300, 9e-281]))[0]
    assert y[0] == 0.0 and np.all(y >= 0.0) and np.all(y <= 1e-140)


def test_exponential_and_erfc(lib):
    x = -np.concatenate([np.linspace(0.0, 700.0, 3001), _range(-60, 9, 500), [0.0]])
    assert _worst(x, _eval(lib, EXP, x)[0], mp.exp) <= 1e-15
    z = np.concatenate([np.linspace(0.0, 6.0, 1201), np.linspace(6.0, 20.0, 401), [1e-300, 1e-8]])
    z = np.concatenate([z, -z])
    y, e = _eval(lib, ERFC, z)
    assert _worst(z, y, mp.erfc) <= 1e-15
    assert _worst(z, e, lambda v: mp.exp(-v * v)) <= 1e-15


def test_ends_of_the_range(lib):
    nan, inf = np.nan, np.inf
    for fn in (RCP, SQRT_RSQRT, SQRT):
        assert np.isnan(_eval(lib, fn, np.array([nan]))[0][0]), fn
    y, e = _eval(lib, ERFC, np.array([0.0, 40.0, -40.0, inf, -inf, 1e200, -1e200, nan]))
    assert list(y[:7]) == [1.0, 0.0, 2.0, 0.0, 2.0, 0.0, 2.0]
    assert list(e[:7]) == [1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0]
    assert np.isnan(y[7]) and np.isnan(e[7])
    y = _eval(lib, EXP, np.array([-800.0, -1e4, -inf]))[0]
    assert np.all(y == 0.0)
