"""How the grid sweeps are shared out over blocks: grids of fewer modes than
one block has threads, row counts that the blocks do not divide, and both
sides of the size from which a resident slot gets more than one block."""
import math

import numpy as np
import pytest

import oracle_py as O
from test_gpu_binning import _rand_grid

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
