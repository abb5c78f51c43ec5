"""The stored rows' splines (csrc/dnu_device.h tri_rows_staged) on knots that are
far from even, compiled for the CPU, against 80-bit elimination: the scans over
the lanes stop after 80 rows, whatever the knots."""
import ctypes as C
import math
import os

import numpy as np
import pytest

from conftest import ROOT
from test_fs_spline import _natural_spline, _p

EMU_LIB = os.path.join(ROOT, "tests", "emu", "_build", "libkn_dnu_emu.so")
X0 = math.log(0.01)


def _knots(name):
    rng = np.random.default_rng(8)
    if name == "growing":        # each interval 5% longer than the one before
        return X0 + np.concatenate([[0.0], np.cumsum(1e-8 * 1.05 ** np.arange(380))])
    if name == "shrinking":
        return X0 + 3.0 - _knots("growing")[::-1] + X0
    if name == "tripling":       # the factors at their largest, in runs over the whole of one window
        h = np.concatenate([1e-9 * 3.0 ** np.arange(18)] * 30)
        return X0 + np.concatenate([[0.0], np.cumsum(h / h.sum() * 4.0)])
    if name == "clusters":
        return np.sort(np.concatenate([np.linspace(X0, -0.1, 300)] + [v + 2e-7 * np.arange(1, 100) for v in (-3.7, -1.9, -0.3)]))
    return np.sort(rng.uniform(X0, 0.0, {"random": 642, "random, two windows": 900}[name]))


@pytest.mark.parametrize("rpw", [1, 2])
@pytest.mark.parametrize("name", ["growing", "shrinking", "tripling", "clusters", "random", "random, two windows"])
def test_rows(kn, name, rpw):
    """A row's error against 80 bits, as h^2 c over the row, within eight times that of the plain elimination in double (the same
    operations, grouped by lanes) or of one rounding of the row."""
    x = np.ascontiguousarray(_knots(name))
    n = len(x)
    assert np.all(np.diff(x) > 0)
    rng = np.random.default_rng(3)
    Y = np.stack([np.exp(x), np.exp(x) * (1 + 0.01 * rng.standard_normal(n)), np.cos(7 * x), (x - X0) ** 3 + 1e-3,
                  1e9 * np.exp(3 * x)])
    c = np.full(Y.shape, np.nan)
    C.CDLL(EMU_LIB).emu_rows_spline(C.c_int(n), C.c_int(len(Y)), C.c_int(rpw), _p(x), _p(Y), _p(c))
    h = np.diff(x)
    hh = np.concatenate([[h[0]], np.maximum(h[1:], h[:-1]), [h[-1]]]) ** 2
    for y, got in zip(Y, c):
        want = _natural_spline(x, y)
        plain = _elimination(x, y)
        e, e0 = (float(np.max(np.abs(v - want) * hh)) for v in (got, plain))
        unit = 2.0 ** -53 * float(np.max(np.abs(y)))
        print("%s: %.2e, plain %.2e, a rounding %.2e" % (name, e, e0, unit))
        assert e <= 8 * max(e0, unit)


def _elimination(x, y):
    n, h = len(x), np.diff(x)
    g, z, al, c = np.zeros(n), np.zeros(n), np.ones(n), np.zeros(n)
    for i in range(1, n - 1):
        rhs = 3 * ((y[i + 1] - y[i]) * (1 / h[i]) - (y[i] - y[i - 1]) * (1 / h[i - 1]))
        al[i] = 2 * (h[i] + h[i - 1]) - (h[i - 1] * g[i - 1] if i > 1 else 0)
        g[i] = h[i] / al[i]
        z[i] = rhs - (g[i - 1] * z[i - 1] if i > 1 else 0)
    for i in range(n - 2, 0, -1):
        c[i] = z[i] / al[i] - g[i] * c[i + 1]
    return c
