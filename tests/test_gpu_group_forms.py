"""The forms a group's launches take by its size, against the per-history
launches (streams mode), which do not change with it: equal bit for bit."""
import ctypes as C
import math

import numpy as np
import pytest

import knhip
from batch_common import Cosmo, compare_adjoint
from dnu_common import synthetic_history

pytestmark = pytest.mark.gpu

HUB = C.CFUNCTYPE(C.c_double, C.c_double, C.c_void_p)


def _merged_and_streams(hists, data, keep):
    B = knhip.Batch(hists, keep=keep)
    for i, (logs, rows, k, init) in enumerate(data):
        B.load(i, logs, rows, k, init)
    g = np.random.default_rng(1).uniform(-1, 1, B.off_k[B.n])
    out = []
    for streams in (0, 4):
        print("group of %d histories, streams %d" % (B.n, streams), flush=True)
        B.set_streams(streams)
        B.solve()
        B.adjoint(g)
        out.append([B.delta_nu(), B._get("dtot_bar", 0, B.off_y[B.n]), B._get("init_bar", 0, B.off_k[B.n]), B.mnu_bar()])
    B.close()
    return out


@pytest.mark.parametrize("steps", [32760, 33000, 40001])
def test_fslength_nodes_by_group_size(kn, torch_cuda, steps):
    """Below, just above and well above the nodes from which the H panels are copied to LDS; chunks that end inside a
    history; tables with a split panel (the density switch of 0.379 eV), without one, and of a stepped H(a) (nodes for the
    second pass, panels whose split records do not all fit)."""
    c = [Cosmo([0.379, 0, 0]), Cosmo([0.0, 0, 0])]
    hub = HUB(lambda a, ctx: 0.1 * math.sqrt(0.3 / a ** 3 + 0.7) *
              (1.3 + 0.3 * math.tanh((math.log(a) - math.log(0.1)) / 0.002)))
    hists, data, left = [], [], steps
    while left > 1:
        na = min(left, [2500, 1111, 129, 3000][len(hists) % 4])
        i = len(hists)
        logs, rows, k, init = synthetic_history(na, 3, 0.6, seed=i, noise=0.0)
        h = c[i % 2].history(3, na, na, 0.6, 0.6, 0.379)
        if i % 5 == 4:
            h.hubble, h.hubble_ctx = C.cast(hub, C.c_void_p).value, None
            h.light, h.delta_nu_prefac = 1.0e5, 1e-9
        hists.append(h)
        data.append((logs, rows, k, init))
        left -= na
    a, b = _merged_and_streams(hists, data, (c, hub))
    assert np.all(np.isfinite(a[0])) and np.all(a[0] != 0)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    for x in c:
        x.free()


@pytest.mark.parametrize("na,noise", [(3, 0.0), (49, 0.1), (400, 0.1), (642, 0.03), (643, 0.03), (1088, 0.0), (1089, 0.0)])
def test_adjoint_by_history_length(kn, torch_cuda, na, noise):
    """The adjoint's windows: shorter than a window's halo, the longest single window, the shortest and longest pair, the
    shortest triple, with a spare step (row stride na + 1); noise per entry makes up to 148 recorded intervals (rounds of
    64, and fewer).  Against the oracle, and merged launches against streams."""
    c = Cosmo([0.3, 0, 0])
    logs, rows, k, init = synthetic_history(na, 3, 0.9, noise=noise)
    h = c.history(3, na, na + 1, 0.9, 0.9, 0.3)
    B = knhip.Batch([h], keep=c)
    B.load(0, logs, rows, k, init)
    g = np.array([0.3, -1.0, 0.7])
    orc = c.oracle(3, logs, rows, init).get_delta_nu_adjoint(0.9, k, 0.3, g)
    assert orc[0] == 0
    out = []
    for streams in (0, 4):
        print("adjoint of %d steps, streams %d" % (na, streams), flush=True)
        B.set_streams(streams)
        B.solve()
        B.adjoint(g)
        out.append((B.delta_nu(0), B.dtot_bar(0, na), B.init_bar(0), B.mnu_bar()[0]))
        compare_adjoint("Na=%d streams %d" % (na, streams), out[-1], orc)
    for x, y in zip(*out):
        assert np.array_equal(x, y)
    B.close()
    c.free()


@pytest.mark.parametrize("rows", [20000, 70000])
def test_rows_per_wavefront(kn, torch_cuda, rows):
    """Histories whose k counts end inside a wavefront's share of rows, of one, two and three windows, in a group with so
    many rows (a history of 3 steps) that wavefronts take 2 and 8 each: equal bit for bit to the same history alone in its
    group, one row per wavefront.  (Noise per entry at 643 and more steps: the oracle's QAG fails too.)"""
    c = Cosmo([0.3, 0, 0])
    hists, data = [], []
    for i, (nk, na) in enumerate([(1, 642), (7, 3), (8, 643), (31, 60), (33, 1089), (65, 1500), (rows, 3)]):
        logs, r, k, init = synthetic_history(na, nk, 0.6, seed=i, noise=0.01 if na < 100 else 0.0)
        hists.append(c.history(nk, na, na + i % 2, 0.6, 0.6, 0.3))
        data.append((logs, r, k, init))
    g = np.random.default_rng(2).uniform(-1, 1, sum(h.nk for h in hists))

    def run(sel):
        B = knhip.Batch([hists[i] for i in sel], keep=c)
        for j, i in enumerate(sel):
            B.load(j, *data[i])
        print("%d rows in %d histories" % (B.off_k[B.n], B.n), flush=True)
        B.solve()
        off = sum(h.nk for h in hists[:sel[0]])
        B.adjoint(g[off:off + B.off_k[B.n]])
        out = [[B.delta_nu(j), B.dtot_bar(j, len(data[i][0])), B.init_bar(j), B.mnu_bar()[j]] for j, i in enumerate(sel)]
        B.close()
        return out

    whole = run(list(range(len(hists))))
    assert all(np.all(np.isfinite(x)) for o in whole for x in o)
    for i in range(len(hists) - 1):
        for x, y in zip(whole[i], run([i])[0]):
            assert np.array_equal(x, y)
    c.free()
