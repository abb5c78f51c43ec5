"""The forms of the free-streaming integral that a launch picks by its stored
steps and species: knots far from the bucket's, stored steps in LDS or in
memory, launches with and without a hybrid species."""
import numpy as np
import pytest

import knhip
from batch_common import Cosmo
from dnu_common import Pair, synthetic_history

pytestmark = pytest.mark.gpu
RTOL = 1e-9   # the bar of the other comparisons with the oracle's QAG


def _steps(na, cluster, amax=0.9):
    """na even steps in log a, or with clusters of many stored steps inside one bucket of the index, smooth in a."""
    logs, rows, k, init = synthetic_history(na, 3, amax, noise=0.0)
    if cluster:
        add = np.concatenate([x + 2e-4 * np.arange(1, 13) for x in (-3.7, -1.9, -0.3)])
        amp = rows[:, 0] / np.exp(logs[0])
        logs = np.sort(np.concatenate([logs, add]))
        rows = np.outer(amp, np.exp(logs))
    return logs, rows, k, init


@pytest.mark.parametrize("hybrid", [None, (500.0, 0.3333)])
@pytest.mark.parametrize("na,cluster", [(2, False), (5, False), (60, True), (300, True), (6144, False), (6145, False)])
def test_stored_steps(kn, torch_cuda, na, cluster, hybrid):
    """Walks of up to twelve knots from the bucket's, the longest history staged in LDS and the next, the linear pair."""
    logs, rows, k, init = _steps(na, cluster)
    P = Pair([0.3, 0, 0], 0.3, len(k), 0.01 + len(logs) / 100.0 + 0.02, hybrid=hybrid)
    P.set_history(logs, rows, init)
    print("get_delta_nu, %d steps%s%s" % (len(logs), ", clusters" * cluster, ", hybrid" if hybrid else ""), flush=True)
    g = P.gpu_get_delta_nu(0.9, k, 0.3)
    rc, o = P.T.get_delta_nu(0.9, k, 0.3)
    assert rc == 0
    e = float(np.max(np.abs(g / o - 1)))
    print("  max rel err vs oracle %.2e" % e)
    assert e < RTOL
    P.free()


@pytest.mark.parametrize("sizes", [(3, 40), (400, 60), (643, 6145)])
def test_group_with_and_without_a_hybrid_history(kn, torch_cuda, sizes):
    """A plain history alone in its group and beside a hybrid one (the launches' other form): the same operations, so
    within their roundings (1e-12 of the largest)."""
    plain, hyb = Cosmo([0.3, 0, 0]), Cosmo([0.3, 0, 0], hybrid=(500.0, 0.3333))
    hists, data = [], []
    for i, na in enumerate(sizes):
        logs, rows, k, init = synthetic_history(na, 5, 0.9, seed=i, noise=0.0)
        hists.append((plain if i == 0 else hyb).history(5, na, na, 0.9, 0.9, 0.3))
        data.append((logs, rows, k, init))
    assert not hists[0].qc > 0 and hists[1].qc > 0
    g = np.random.default_rng(3).uniform(-1, 1, 5)
    out = []
    for n in (1, 2):
        B = knhip.Batch(hists[:n], keep=(plain, hyb))
        for i in range(n):
            B.load(i, *data[i])
        print("group of %d, steps %s" % (n, sizes), flush=True)
        B.solve()
        B.adjoint(np.concatenate([g] * n))
        out.append((B.delta_nu(0), B.dtot_bar(0, sizes[0]), B.init_bar(0), B.mnu_bar()[0]))
        B.close()
    for x, y in zip(*out):
        assert np.max(np.abs(x - y)) <= 1e-12 * np.max(np.abs(x))
    plain.free()
    hyb.free()
