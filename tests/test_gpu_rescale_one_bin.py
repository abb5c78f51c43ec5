"""A ratio table of one bin: its ratio at every k, whatever its log k is."""
import math

import numpy as np
import pytest

from test_gpu_binning import _rand_grid

pytestmark = pytest.mark.gpu

BOX = 512000.0


@pytest.mark.parametrize("N", [6, 130])
@pytest.mark.parametrize("logk", [-9.0, 0.0, math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("box", [BOX, math.nan])
def test_one_bin(kn, torch_cuda, N, logk, box):
    """Every mode but k = 0 times 1 + norm ratio, rounded once in the factor and once in the product."""
    torch = torch_cuda
    print("one bin", N, logk, box, flush=True)
    F = _rand_grid(N, 3, 2)
    d, tab = torch.from_numpy(F).cuda(), torch.tensor([logk, 0.37], dtype=torch.float64).cuda()
    assert kn.kn_rescale_device(d.data_ptr(), N, 0, 2, box, tab.data_ptr(), tab.data_ptr() + 8, 1, 0.21, None) == 0
    got = d.cpu().numpy()
    assert got[0, 0, 0] == F[0, 0, 0]
    want = F * (1 + 0.21 * 0.37)
    want[0, 0, 0] = F[0, 0, 0]
    np.testing.assert_allclose(got.view(np.float64), want.view(np.float64), rtol=4.5e-16, atol=0)
