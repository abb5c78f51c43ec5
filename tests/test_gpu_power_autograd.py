"""The device-resident spectrum and its adjoint (kn_power_spectrum_device,
kn_power_spectrum_adjoint_device) through the autograd function, against
total_powerspectrum and the oracle's adjoint."""
import ctypes as C

import numpy as np
import pytest

import knhip
import oracle_py as O
from test_gpu_binning import _rand_grid

pytestmark = pytest.mark.gpu


# empty bins at (8, 300) and (32, 20000) (tables in global memory); one block of 1024 threads takes 1, 2 and 20 bins each
@pytest.mark.parametrize("N,nrbins", [(8, 12), (8, 300), (9, 5), (15, 1025), (32, 40), (32, 20000)])
@pytest.mark.parametrize("own_stream", [False, True])
def test_spectrum_and_gradient(kn, torch_cuda, N, nrbins, own_stream):
    torch = torch_cuda
    F = _rand_grid(N, seed=N)
    F[0, 0, 0] = N ** 3 * (1 - 0.2j)
    on, op, _, _ = O.total_powerspectrum(F, nrbins)
    g = np.random.default_rng(N).uniform(-1, 1, on)
    rc, ofb = O.bin_power_adjoint(F, nrbins, g)
    assert rc == 0
    host = torch.from_numpy(np.ascontiguousarray(F).view(np.float64).reshape(N, N, N // 2 + 1, 2))
    st = torch.cuda.Stream() if own_stream else torch.cuda.current_stream()
    print("spectrum and gradient", N, nrbins, own_stream, flush=True)
    fn = knhip.power_spectrum_function()
    with torch.cuda.stream(st):
        field = host.cuda().requires_grad_(True)
        power = fn.apply(field, nrbins)
        first = power.detach().cpu().numpy()
        power = power * torch.from_numpy(g).cuda()
        power.mul_(1.0)
        power.sum().backward()          # an expanded gradient of the product, and of the spectrum g
        bar = field.grad.cpu().numpy()
    assert len(first) == on
    np.testing.assert_allclose(first, op[:on], rtol=1e-12)
    e = np.max(np.abs(bar.view(np.complex128).reshape(F.shape) - ofb)) / np.max(np.abs(ofb))
    print("  max err %.2e of max |dL/dF|" % e)
    assert e < 1e-12


def test_output_is_the_callers(kn, torch_cuda):
    """The spectrum may be changed in place, take an expanded gradient, and a wrong length is refused."""
    torch = torch_cuda
    F = _rand_grid(8, seed=1)
    F[0, 0, 0] = 512.0
    fn = knhip.power_spectrum_function()
    field = torch.from_numpy(np.ascontiguousarray(F).view(np.float64).reshape(8, 8, 5, 2)).cuda().requires_grad_(True)
    out = []
    for scale in (False, True):
        p = fn.apply(field, 12)
        if scale:
            p *= 2.0
        (bar,) = torch.autograd.grad(p.sum(), field)
        out.append(bar)
    assert torch.equal(2.0 * out[0], out[1])
    g = torch.ones(p.numel() + 1, dtype=torch.float64, device="cuda")
    assert kn.kn_power_spectrum_adjoint_device(field.data_ptr(), 8, 12, 0, 8, g.data_ptr(), g.data_ptr(), p.numel() + 1,
                                               out[0].data_ptr(), None) == 3002
    assert kn.kn_power_spectrum_adjoint_device(field.data_ptr(), 8, 12, 2, 6, g.data_ptr(), g.data_ptr(), p.numel(),
                                               out[0].data_ptr(), None) == 3002
