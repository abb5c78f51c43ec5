"""The fslength table's spline (csrc/dnu_device.h uniform_spline_wave), compiled
for the CPU, against the natural spline on the same knots in 80-bit arithmetic:
knots far apart, where its factors are constants, and so close that their
rounding shows in their spacings."""
import ctypes as C
import math
import os

import numpy as np
import pytest

from conftest import ROOT

EMU_LIB = os.path.join(ROOT, "tests", "emu", "_build", "libkn_dnu_emu.so")
LD = np.longdouble


def _p(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def _natural_spline(x, y):
    x, y = x.astype(LD), y.astype(LD)
    n, h = len(x), np.diff(x)
    g, z, al, c = np.zeros(n, LD), np.zeros(n, LD), np.ones(n, LD), np.zeros(n, LD)
    dy = np.diff(y) / h
    for i in range(1, n - 1):
        al[i] = 2 * (h[i] + h[i - 1]) - (h[i - 1] * g[i - 1] if i > 1 else 0)
        g[i] = h[i] / al[i]
        z[i] = 3 * (dy[i] - dy[i - 1]) - (g[i - 1] * z[i - 1] if i > 1 else 0)
    for i in range(n - 2, 0, -1):
        c[i] = z[i] / al[i] - g[i] * c[i + 1]
    return c


def _values(x, y, c, t):
    x, y, c = x.astype(LD), y.astype(LD), c.astype(LD)
    h, dy = np.diff(x), np.diff(y)
    b, d, dx = dy / h - h * (c[1:] + 2 * c[:-1]) / 3, (c[1:] - c[:-1]) / (3 * h), LD(t) * h
    return y[:-1] + dx * (b + dx * (c[:-1] + dx * d))


# without those that end past a = 1.6, or whose knots coincide
CASES = [(x0, span, n) for x0 in (math.log(0.01), math.log(0.4))
         for span in (1e-12, 1e-10, 1e-8, 1e-6, 2e-5, 1e-4, 1.2e-3, 0.1, 4.5) for n in (32, 80, 642, 643, 1600, 5000)
         if x0 + span <= 0.5 and span >= 40 * n * 2.0 ** -52 * abs(x0)]


@pytest.mark.parametrize("x0,span,n", CASES)
def test_spline_values(kn, x0, span, n):
    """A slope is formed with two or three roundings, and a value takes at most h (2 + 2) of neighbouring slopes' errors, twice
    (right-hand side and coefficient): 16 roundings of the largest step of y, whatever the span.  (The sides of
    h = 2^-25 |x| at 32, 80 and 642 knots lie at spans of 4e-6, 1.1e-5 and 9e-5 from 0.01.)"""
    xa = x0 + span
    x = np.array([x0 + i * (xa - x0) / (n - 1.0) for i in range(n)])
    f = lambda t: 2 * np.exp(LD(0.5) * t.astype(LD))
    y = (f(np.array([xa]))[0] - f(x)).astype(np.float64)   # falls to 0 at the last knot, as a length to come does
    L = C.CDLL(EMU_LIB)
    xs, c = np.zeros(n), np.full(n, np.nan)
    L.emu_fs_spline(C.c_double(x0), C.c_double(xa), C.c_int(n), _p(y), _p(xs), _p(c))
    assert np.array_equal(xs, x) and c[0] == 0.0 and c[-1] == 0.0
    want = _natural_spline(x, y)
    err = max(float(np.max(np.abs(_values(x, y, c, t) - _values(x, y, want, t)))) for t in (0.2, 0.5, 0.8))
    unit = 2.0 ** -53 * float(np.max(np.abs(np.diff(y))))
    print("n %d span %.0e: %.2f roundings of a step" % (n, span, err / unit))
    assert err <= 16 * unit
