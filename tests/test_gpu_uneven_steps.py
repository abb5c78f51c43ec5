"""Forward and adjoint of histories whose stored steps are far from even, in one
window and in two, against the oracle."""
import math

import numpy as np
import pytest

import knhip
from batch_common import Cosmo, compare_adjoint
from dnu_common import synthetic_history

pytestmark = pytest.mark.gpu

X0, X1 = math.log(0.01), math.log(0.9)


def _steps(name):
    if name == "growing":
        h = 1.03 ** np.arange(400)
    elif name == "shrinking":
        h = 1.03 ** np.arange(400)[::-1]
    elif name == "tripling":
        h = np.concatenate([3.0 ** np.arange(8)] * 20)
    else:
        h = np.random.default_rng(6).uniform(0.05, 1.0, {"random": 640, "two windows": 800}[name])
    x = X0 + (X1 - X0) * np.concatenate([[0.0], np.cumsum(h / h.sum())])
    x[-1] = X1
    return x


@pytest.mark.parametrize("name", ["growing", "shrinking", "tripling", "random", "two windows"])
def test_uneven_steps(kn, torch_cuda, name):
    """The bar of the other comparisons with the oracle, merged launches and streams."""
    x = _steps(name)
    na = len(x)
    c = Cosmo([0.3, 0, 0])
    _, rows, k, init = synthetic_history(na, 3, 0.9, noise=0.0)
    rows = np.outer(rows[:, 0], np.exp(x - x[0])) * (1 + 0.02 * np.sin(9 * x))
    B = knhip.Batch([c.history(3, na, na, 0.9, 0.9, 0.3)], keep=c)
    B.load(0, x, rows, k, init)
    g = np.array([0.3, -1.0, 0.7])
    orc = c.oracle(3, x, rows, init).get_delta_nu_adjoint(0.9, k, 0.3, g)
    assert orc[0] == 0
    for streams in (0, 2):
        print("uneven steps", name, streams, flush=True)
        B.set_streams(streams)
        B.solve()
        B.adjoint(g)
        compare_adjoint("%s, streams %d" % (name, streams), (B.delta_nu(0), B.dtot_bar(0, na), B.init_bar(0),
                                                             B.mnu_bar()[0]), orc)
    B.close()
    c.free()
