"""The rescale sweep's log(sqrt(k2)) (csrc/half_log.h), compiled for the CPU,
against the 80-bit logarithm."""
import ctypes as C
import os

import numpy as np
import pytest

from conftest import ROOT

EMU_LIB = os.path.join(ROOT, "tests", "emu", "_build", "libkn_dnu_emu.so")


@pytest.mark.parametrize("which", ["small", "powers", "edges", "any"])
def test_half_log(kn, which):
    """Half a unit in the last place of the result, as half of a correctly rounded log(k2), plus 2^-56 for the series (2e-18),
    the table's residue (2^-58) and the rounding of what is added last (below 2e-3: 2^-62)."""
    rng = np.random.default_rng(0)
    top = 2 ** 31 - 1
    k2 = {"small": np.arange(1, 300001),
          "powers": np.concatenate([2 ** np.arange(0, 31) + d for d in (-1, 0, 1)]),
          # both sides of every interval of the table, at all exponents that resolve it
          "edges": np.concatenate([(128 + np.arange(128)) * 2 ** e + d for e in range(0, 24) for d in (-1, 0, 1)]),
          "any": np.concatenate([rng.integers(1, top + 1, 200000), np.exp(rng.uniform(0, np.log(top), 200000)).astype(int)])}[which]
    k2 = np.unique(k2[(k2 >= 1) & (k2 <= top)]).astype(np.int32)
    L = C.CDLL(EMU_LIB)
    out = np.zeros(len(k2))
    L.emu_half_log(C.c_int(len(k2)), k2.ctypes.data_as(C.POINTER(C.c_int)), out.ctypes.data_as(C.POINTER(C.c_double)))
    want = np.log(k2.astype(np.longdouble)) / 2
    err = np.abs(out - want).astype(float)
    bound = 0.5 * np.spacing(np.maximum(np.abs(out), 2.0 ** -30)) + 2.0 ** -56
    print("%s: worst %.3e, of its bound %.3f" % (which, err.max(), (err / bound).max()))
    assert np.all(err <= bound)
