"""specialJ's fit and its power x^4.1811 (csrc/dnu_device.h), compiled for the
CPU, against 80-bit arithmetic, at and beyond the ends of the power's table."""
import ctypes as C
import os

import numpy as np
import pytest

from conftest import ROOT

EMU_LIB = os.path.join(ROOT, "tests", "emu", "_build", "libkn_dnu_emu.so")
LD = np.longdouble
P = LD(4.1811)  # the double


def _p(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def _points():
    rng = np.random.default_rng(1)
    edges = 1 + np.arange(128) / 128
    m = np.concatenate([edges, np.nextafter(edges, 0), np.nextafter(edges, 3), edges + 1 / 256, rng.uniform(1, 2, 4000)])
    return np.concatenate([m, m * 2.0 ** rng.integers(-64, 65, len(m)), m * 2.0 ** -64, m[m < 2] * 2.0 ** 64,
                           2.0 ** np.arange(-64, 65)])


def test_power(kn):
    """Two units in the last place: table entries and the fused sum half a unit each, the last product half a unit."""
    L = C.CDLL(EMU_LIB)
    x = _points()
    x = x[(x >= 2.0 ** -64) & (x < 2.0 ** 65)]
    out = np.zeros(len(x))
    L.emu_pow_fit(C.c_int(len(x)), _p(x), _p(out))
    err = np.abs(out / x.astype(LD) ** P - 1).astype(float)
    print("x^4.1811: worst %.2f units of 2^-52" % (err.max() * 2 ** 52))
    assert err.max() <= 2 * 2.0 ** -52
    far = np.array([5e-324, 1e-300, 2.0 ** -70, 2.0 ** 70, 1e300])
    out = np.zeros(len(far))
    L.emu_pow_fit(C.c_int(len(far)), _p(far), _p(out))
    assert np.all(np.isfinite(out)) and np.all(out > 0)


@pytest.mark.parametrize("lo,hi", [(-290, -41), (-41, -19), (-20, -3), (-3, 3), (3, 18)])
def test_fit_and_derivative(kn, lo, hi):
    """N, D and their derivatives carry at most eight roundings each, the two products differ by a factor of two or more
    (so that their difference magnifies them by at most 3.1), the square and the quotient three: 1e-14 in all; the value
    N / D twice eight and one: 2e-15."""
    L = C.CDLL(EMU_LIB)
    x = 10.0 ** np.random.default_rng(2).uniform(lo, hi, 3000)
    J, Jx, Jq = np.zeros(len(x)), np.zeros(len(x)), np.ones(len(x))
    L.emu_specialJ_d(C.c_int(len(x)), _p(x), C.c_double(0.0), C.c_double(0.0), _p(J), _p(Jx), _p(Jq))
    t = x.astype(LD)
    c = [LD(v) for v in (0.0168, 0.0407, 2.1734, 1.6787, 0.1467)]
    N, D = 1 + c[0] * t ** 2 + c[1] * t ** 4, 1 + c[2] * t ** 2 + c[3] * t ** P + c[4] * t ** 8
    Nx = 2 * c[0] * t + 4 * c[1] * t ** 3
    Dx = 2 * c[2] * t + c[3] * P * t ** (P - 1) + 8 * c[4] * t ** 7
    want = (Nx * D - N * Dx) / (D * D)
    ev, ed = float(np.max(np.abs(J / (N / D) - 1))), float(np.max(np.abs(Jx / want - 1)))
    print("1e%d..1e%d: value %.2e, derivative %.2e" % (lo, hi, ev, ed))
    assert ev < 2e-15 and ed < 1e-14
    assert np.all(Jq == 0.0)
