"""The grid sweeps at both sides of the tile counts at which their launches
change: a tile per block, or blocks that take tiles in turn; own bin sums per
wavefront, or shared ones.  (256 CUs: 512 resident blocks of the rescale, one
per CU with more than 80 KB of tables; 512 and 768 tiles of the bin sweep.)"""
import math

import numpy as np
import pytest

import oracle_py as O
from test_gpu_binning import _rand_grid

pytestmark = pytest.mark.gpu

BOX = 512000.0
# rows of fewer than 64 modes, tiles of 512: 488 and 513, 744 and 777 tiles; longer rows, tiles of 1024: 512 and 520, 764 and
# 772 tiles; 252 and 260
SIZES = [(79, 0, 79), (80, 0, 80), (91, 0, 91), (92, 0, 92), (126, 3, 65), (126, 3, 66), (126, 0, 97), (126, 0, 98),
         (128, 0, 31), (128, 1, 32)]


@pytest.mark.parametrize("N,start,nslab", SIZES)
@pytest.mark.parametrize("nb", [19, 2600])
def test_rescale_tiles(kn, torch_cuda, N, start, nslab, nb):
    """1e-14, as the sweeps' other tests (the ratio's slope is below one)."""
    torch = torch_cuda
    print("rescale tiles", N, start, nslab, nb, flush=True)
    F = _rand_grid(N, 5, nslab)
    lk = np.log(np.geomspace(2 * math.pi / BOX, math.sqrt(3) * math.pi * N / BOX, nb))
    rt = np.sin(lk)
    d, tab = torch.from_numpy(F).cuda(), torch.from_numpy(np.concatenate([lk, rt])).cuda()
    assert kn.kn_rescale_device(d.data_ptr(), N, start, nslab, BOX, tab.data_ptr(), tab.data_ptr() + 8 * nb, nb, 0.07,
                                None) == 0
    torch.cuda.synchronize()
    rc, W = O.rescale(F, BOX, lk, rt, 0.07, start)
    assert rc == 0
    np.testing.assert_allclose(d.cpu().numpy().view(np.float64), W.view(np.float64), rtol=1e-14, atol=0)


@pytest.mark.parametrize("N,start,nslab", SIZES)
@pytest.mark.parametrize("nb", [20, 200, 2000])
def test_bin_tiles(kn, torch_cuda, N, start, nslab, nb):
    """1e-12, as the sums' other tests (added in another order)."""
    torch = torch_cuda
    print("bin tiles", N, start, nslab, nb, flush=True)
    F = _rand_grid(N, 7, nslab)
    d, want = torch.from_numpy(F).cuda(), O.bin_sums(F, nb, start)[0]
    for fn in (kn.kn_bin_power_device, kn.kn_bin_power_device_noalloc):
        p = torch.full((nb + 1,), -1.0, dtype=torch.float64, device="cuda")
        assert fn(d.data_ptr(), N, nb, start, nslab, p.data_ptr(), p.data_ptr() + 8 * nb, None) == 0
        np.testing.assert_allclose(p.cpu().numpy()[:nb], want, rtol=1e-12, atol=0)
