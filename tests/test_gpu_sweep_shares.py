"""How the grid sweeps are shared out over blocks: grids of fewer modes than
one block has threads, row counts that the blocks do not divide, and both
sides of the size from which a resident slot gets more than one block."""
import math

import numpy as np
import pytest

import oracle_py as O
from test_gpu_binning import _rand_grid, check_against_oracle

pytestmark = pytest.mark.gpu

BOX = 512000.0


@pytest.mark.parametrize("N,start,nslab", [(3, 0, 1), (4, 2, 1), (31, 7, 5), (64, 0, 64), (250, 100, 37), (256, 0, 256),
                                           (322, 0, 322), (324, 0, 324)])
@pytest.mark.parametrize("green", [False, True])
def test_rescale_shares(kn, torch_cuda, N, start, nslab, green):
    """To 1e-14, as the sweeps' other tests: one rounding of the factor, one of the product."""
    torch = torch_cuda
    print("rescale shares", N, start, nslab, green, flush=True)
    F = _rand_grid(N, 5, nslab)
    nb = 19
    lk = np.log(np.geomspace(2 * math.pi / BOX, math.sqrt(3) * math.pi * N / BOX, nb))
    rt = np.random.default_rng(2).uniform(0, 1, nb)
    d, tab = torch.from_numpy(F).cuda(), torch.from_numpy(np.concatenate([lk, rt])).cuda()
    args = (d.data_ptr(), N, start, nslab, BOX, tab.data_ptr(), tab.data_ptr() + 8 * nb, nb, 0.07)
    asmth = 1.25 * BOX / N
    rc = kn.kn_rescale_green_device(*args, asmth, None) if green else kn.kn_rescale_device(*args, None)
    torch.cuda.synchronize()
    rc2, W = O.rescale(F, BOX, lk, rt, 0.07, start)
    if green:
        W = O.green(W, BOX, asmth, start)
    assert rc == 0 and rc2 == 0
    np.testing.assert_allclose(d.cpu().numpy().view(np.float64), W.view(np.float64), rtol=1e-14, atol=0)


@pytest.mark.parametrize("N,start,nslab,nb", [(4, 0, 4, 15), (5, 3, 1, 7), (33, 0, 33, 9), (96, 0, 96, 96), (192, 0, 192, 64),
                                              (250, 100, 37, 64), (250, 0, 250, 1000), (64, 0, 64, 12000), (125, 3, 122, 40),
                                              (126, 1, 5, 2), (127, 120, 7, 33), (128, 0, 128, 1), (200, 0, 200, 13500),
                                              (40, 0, 40, 15000), (160, 1, 159, 15000)])
def test_bin_shares(kn, torch_cuda, N, start, nslab, nb):
    """One block and one partial row, a tile per block, all resident blocks; rows of just under and over 64 modes; one bin,
    and the bin counts where own sums, copies, LDS tables and one-wavefront blocks begin and end
    (counts equal, sums to 1e-12 as the other tests of the sums: they are added in another order)."""
    torch = torch_cuda
    F = _rand_grid(N, 7, nslab)
    if start == 0:
        check_against_oracle(kn, torch, F, nb)
        return
    d, p = torch.from_numpy(F).cuda(), torch.full((nb + 1,), -1.0, dtype=torch.float64, device="cuda")
    for fn in (kn.kn_bin_power_device, kn.kn_bin_power_device_noalloc):
        print("bin shares", N, start, nslab, nb, flush=True)
        assert fn(d.data_ptr(), N, nb, start, nslab, p.data_ptr(), p.data_ptr() + 8 * nb, None) == 0
        got = p.cpu().numpy()
        want = O.bin_sums(F, nb, start)[0]
        np.testing.assert_allclose(got[:nb], want, rtol=1e-12, atol=0)
        assert got[nb] == 0.0


@pytest.mark.parametrize("N,nb", [(8, 10), (32, 1500), (36, 12000), (64, 64), (130, 20), (256, 32)])
def test_bin_sums_repeat(kn, torch_cuda, N, nb):
    """Own bin sums per wavefront (small grids, and few bins at any size), and small grids with one wavefront per block for
    want of LDS: the same bits on every run."""
    torch = torch_cuda
    print("bin repeat", N, nb, flush=True)
    d = torch.from_numpy(_rand_grid(N, 9)).cuda()
    out = []
    for _ in range(4):
        p = torch.zeros(nb + 1, dtype=torch.float64, device="cuda")
        assert kn.kn_bin_power_device(d.data_ptr(), N, nb, 0, N, p.data_ptr(), p.data_ptr() + 8 * nb, None) == 0
        out.append(p.cpu().numpy())
    assert all(np.array_equal(out[0], o) for o in out[1:])


@pytest.mark.parametrize("N", [6, 124, 125, 126, 250])
def test_rescale_log_k(kn, torch_cuda, N):
    """A ratio equal to log k turns each mode's factor into 1 + norm log k.  The bound: log k (below 12) within 1.8e-15 of
    its logarithm's table and three roundings at 12 (0.9e-15 each), norm times that, over a factor of 1.9 or more."""
    torch = torch_cuda
    print("rescale log k", N, flush=True)
    lk = np.array([math.log(2 * math.pi / BOX) - 1e-3, math.log(math.sqrt(3) * math.pi * N / BOX) + 1e-3])
    tab, norm = torch.from_numpy(np.concatenate([lk, lk])).cuda(), 0.5
    d = torch.ones((N, N, N // 2 + 1), dtype=torch.complex128, device="cuda")
    assert kn.kn_rescale_device(d.data_ptr(), N, 0, N, BOX, tab.data_ptr(), tab.data_ptr() + 16, 2, norm, None) == 0
    i = np.arange(N)
    kv = np.where(i <= N // 2, i, i - N)
    k2 = (kv[:, None, None] ** 2 + kv[None, :, None] ** 2 + np.arange(N // 2 + 1)[None, None, :] ** 2).astype(np.longdouble)
    k2[0, 0, 0] = 1
    s = 1 + np.longdouble(norm) * (np.log(k2) / 2 + np.log(2 * np.longdouble(math.pi) / BOX))
    got = d.cpu().numpy().real
    assert got[0, 0, 0] == 1.0
    e = np.abs(got / s - 1)
    e[0, 0, 0] = 0
    print("  worst %.2e" % float(e.max()))
    assert float(e.max()) < norm * 4.5e-15 / 1.9 + 2.3e-16


@pytest.mark.parametrize("nb", [1, 2, 700, 4050, 5000])
def test_rescale_table_sizes(kn, torch_cuda, nb):
    """One bin to the largest tables (a bucket per bin in place of four from 4045 bins on), unevenly spaced; past the
    limit the call is refused as ever."""
    torch = torch_cuda
    print("rescale table", nb, flush=True)
    N, rng = 130, np.random.default_rng(nb)
    F = _rand_grid(N, 11, 9)
    lk = np.sort(rng.uniform(math.log(math.pi / BOX), math.log(2 * math.pi * N / BOX), nb)) if nb > 1 else np.array([-9.0])
    rt = rng.uniform(-1, 1, nb)
    d, tab = torch.from_numpy(F).cuda(), torch.from_numpy(np.concatenate([lk, rt])).cuda()
    assert kn.kn_rescale_device(d.data_ptr(), N, 0, 9, BOX, tab.data_ptr(), tab.data_ptr() + 8 * nb, nb, 0.05, None) == 0
    torch.cuda.synchronize()
    rc, W = O.rescale(F, BOX, lk, rt, 0.05, 0)
    assert rc == 0
    # a segment of width h turns an error of 4e-15 in log k into one of norm |d ratio| 4e-15 / h in the factor
    h = max(np.min(np.diff(lk)), 1e-9) if nb > 1 else 1.0
    np.testing.assert_allclose(d.cpu().numpy().view(np.float64), W.view(np.float64), rtol=1e-14 + 0.05 * 2 * 4e-15 / h, atol=0)
    assert kn.kn_rescale_device(d.data_ptr(), N, 0, 9, BOX, tab.data_ptr(), tab.data_ptr(), 5200, 0.05, None) == 3002
