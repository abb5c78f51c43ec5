"""specialJ's table-driven power x^4.1811 (kn_powtab.h, dnu_device.h pow_fit),
its tables and series restated in exact arithmetic: within 2 units in the last
place at interval edges, centres, binary exponents' ends and random x."""
import os
import re

import numpy as np
import pytest

from conftest import ROOT

mp = pytest.importorskip("mpmath").mp


def _tables():
    src = open(os.path.join(ROOT, "kspace-neutrinos_amd", "csrc", "kn_powtab.h")).read()
    tab, ex = (np.array([float.fromhex(v) for v in re.findall(r"-?0x[0-9a-f.]+p[+-]\d+", part)])
               for part in re.findall(r"= \{(.*?)\};", src, re.S))
    a = [float.fromhex(v) for v in re.findall(r"#define KN_POW_A\d (\S+)", src)]
    return tab.reshape(-1, 2), ex, a


def test_power_table():
    mp.dps = 40
    tab, ex, a = _tables()
    assert tab.shape == (128, 2) and len(ex) == 129 and len(a) == 5
    rng = np.random.default_rng(0)
    edges = 1 + np.arange(128) / 128
    m = np.concatenate([edges, np.nextafter(edges[1:], 0), [np.nextafter(2.0, 0)], edges + 1 / 256, rng.uniform(1, 2, 300)])
    x = np.concatenate([m, m * 2.0 ** rng.integers(-64, 65, len(m)), 2.0 ** np.arange(-64, 65)])
    p = mp.mpf(4.1811)
    for v in x:
        mant, e = np.frexp(v)
        mant, e = 2 * mant, e - 1
        r_j, t = tab[int((mant - 1) * 128)]
        r = float(mp.mpf(mant) * mp.mpf(r_j) - 1)
        assert abs(r) <= 2.0 ** -8 + 2.0 ** -50
        q = mp.mpf(0)
        for c in reversed(a):   # each step rounded once, as the fused operations
            q = mp.mpf(float(q * r + mp.mpf(c)))
        q = float(q * r)
        got = mp.mpf(float(mp.mpf(t) * q + mp.mpf(t))) * mp.mpf(ex[e + 64])
        # table entries and fused sum half a unit each, the last product half a unit: four halves of 2^-52 at most
        assert abs(mp.mpf(float(got)) / mp.mpf(float(v)) ** p - 1) <= 2 * 2.0 ** -52
