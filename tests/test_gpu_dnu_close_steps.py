"""Stored steps so close to the starting scale factor that the fslength table's
knots show their rounding, and just far enough that they do not: the integral
against its limit for a short interval."""
import ctypes as C
import math

import numpy as np
import pytest

import knhip
from batch_common import Cosmo
from dnu_common import synthetic_history

pytestmark = pytest.mark.gpu

HUB = C.CFUNCTYPE(C.c_double, C.c_double, C.c_void_p)


@pytest.mark.parametrize("streams", [0, 2])
@pytest.mark.parametrize("na", [3, 5, 60])
@pytest.mark.parametrize("span", [1e-10, 1e-8, 1e-6])
def test_short_interval(kn, torch_cuda, span, na, streams):
    """H = a^-3/2: over [log T0, log T0 + span] the length to come is light a^-1/2 (xa - x), the rows are constant and specialJ
    is 1 - 2.2 (k fsl / m)^2, so the integral is light S span^2 / 2 (a H = a^-1/2) to relative 2 span + 1e-12 for specialJ,
    and to 4 units in the last place of log T0 over span for the interval's own ends."""
    T0, light, prefac, S = 0.01, 1.0, 1e30, 3.0
    hub = HUB(lambda a, ctx: a ** -1.5)
    c = Cosmo([0.3, 0, 0])
    _, _, k, init = synthetic_history(na, 4, 0.9)
    x0 = math.log(T0)
    logs = x0 + span * np.arange(na) / (na - 1.0)
    h = c.history(4, na, na, float(np.exp(logs[-1])), 0.9, 0.3)
    h.hubble, h.hubble_ctx, h.light, h.delta_nu_prefac = C.cast(hub, C.c_void_p).value, None, light, prefac
    B = knhip.Batch([h], keep=(c, hub))
    xa = math.log(h.a)
    logs[-1] = max(logs[-1], xa)   # log(exp(log a)) may lie a rounding further on
    B.load(0, logs, np.full((4, na), S), 1e-3 * k / k[-1], 0.0 * init)
    B.set_streams(streams)
    print("short interval", span, na, streams, flush=True)
    B.solve()
    d = xa - x0
    want = prefac * light * S * T0 ** -0.5 * T0 ** 0.5 * d * d / 2
    e = float(np.max(np.abs(B.delta_nu(0) / want - 1)))
    print("  rel err %.2e" % e)
    assert e < 2 * span + 1e-12 + 4 * 2.0 ** -52 * abs(x0) / span
    B.close()
    c.free()
