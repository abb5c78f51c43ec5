"""The device-resident spectrum and its adjoint beside other calls of the same
geometry on other streams: every call's results are those it gives alone."""
import ctypes as C

import numpy as np
import pytest

import knhip
import oracle_py as O
from test_gpu_binning import _rand_grid

pytestmark = pytest.mark.gpu


def _grids(torch, N, n):
    out = []
    for i in range(n):
        F = _rand_grid(N, seed=20 + i)
        F[0, 0, 0] = N ** 3 * (1 + 0.1j * i)
        out.append((F, torch.from_numpy(np.ascontiguousarray(F).view(np.float64).reshape(N, N, N // 2 + 1, 2)).cuda()))
    return out


@pytest.mark.parametrize("N,nb", [(24, 24), (130, 40), (130, 1500)])
def test_other_calls_of_a_geometry(kn, torch_cuda, N, nb):
    """Spectra and gradients of one field by the device forms on one stream, bin sums (and gradients) of another field by
    kn_bin_power_device and kn_bin_power_adjoint on a second stream, all in flight together: 1e-12 of the oracle, as the
    calls alone (tests of the sums: added in another order)."""
    torch = torch_cuda
    (Fa, a), (Fb, b) = _grids(torch, N, 2)
    wantA, wantB = O.total_powerspectrum(Fa, nb), O.bin_sums(Fb, nb, 0)[0]
    on = wantA[0]
    gb = np.random.default_rng(5).uniform(-1, 1, on)
    barA, barB = O.bin_power_adjoint(Fa, nb, gb), O.bin_power_adjoint(Fb, nb, gb[::-1].copy())
    assert barA[0] == 0 and barB[0] == 0
    g, gr = torch.from_numpy(gb).cuda(), gb[::-1].copy()
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    print("calls of one geometry on two streams", N, nb, flush=True)
    reps, n = 12, C.c_int()
    power = torch.zeros((reps, nb), dtype=torch.float64, device="cuda")
    bars = [torch.empty_like(a) for _ in range(reps)]
    sums = torch.zeros((reps, nb + 1), dtype=torch.float64, device="cuda")
    barb = torch.empty_like(b)
    torch.cuda.synchronize()
    for r in range(reps):
        assert kn.kn_power_spectrum_device(a.data_ptr(), N, nb, 0, N, power[r].data_ptr(), C.byref(n), s1.cuda_stream) == 0
        assert kn.kn_bin_power_device(b.data_ptr(), N, nb, 0, N, sums[r].data_ptr(), sums[r].data_ptr() + 8 * nb,
                                      s2.cuda_stream) == 0
        assert kn.kn_power_spectrum_adjoint_device(a.data_ptr(), N, nb, 0, N, power[r].data_ptr(), g.data_ptr(), on,
                                                   bars[r].data_ptr(), s1.cuda_stream) == 0
        if r % 3 == 2:   # waits for its own stream; the first stream's gradient may still be under way
            assert kn.kn_bin_power_adjoint(b.data_ptr(), N, nb, 0, N, gr.ctypes.data_as(knhip.dp), on, barb.data_ptr(),
                                           s2.cuda_stream) == 0
            e = np.max(np.abs(barb.cpu().numpy().view(np.complex128).reshape(Fb.shape) - barB[1]))
            assert e < 1e-12 * np.max(np.abs(barB[1]))
    torch.cuda.synchronize()
    assert n.value == on
    for r in range(reps):
        np.testing.assert_allclose(power[r].cpu().numpy()[:on], wantA[1][:on], rtol=1e-12)
        np.testing.assert_allclose(sums[r].cpu().numpy()[:nb], wantB, rtol=1e-12, atol=0)
        e = np.max(np.abs(bars[r].cpu().numpy().view(np.complex128).reshape(Fa.shape) - barA[1]))
        assert e < 1e-12 * np.max(np.abs(barA[1]))


def test_two_streams_and_autograd(kn, torch_cuda):
    """The autograd function on two streams without a host wait between, forward and backward: each field's own result."""
    torch = torch_cuda
    N, nb = 64, 48
    fields = _grids(torch, N, 2)
    fn = knhip.power_spectrum_function()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    print("autograd on two streams", flush=True)
    got = [[], []]
    for r in range(6):
        for i in (0, 1):
            with torch.cuda.stream(streams[i]):
                x = fields[i][1].detach().requires_grad_(True)
                p = fn.apply(x, nb)
                (bar,) = torch.autograd.grad((p * (1.0 + r)).sum(), x)
                got[i].append((p.detach(), bar))
    torch.cuda.synchronize()
    for i in (0, 1):
        on, op, _, _ = O.total_powerspectrum(fields[i][0], nb)
        rc, ob = O.bin_power_adjoint(fields[i][0], nb, np.ones(on))
        assert rc == 0
        for r, (p, bar) in enumerate(got[i]):
            np.testing.assert_allclose(p.cpu().numpy(), op[:on], rtol=1e-12)
            e = np.max(np.abs(bar.cpu().numpy().view(np.complex128).reshape(ob.shape) / (1.0 + r) - ob))
            assert e < 1e-12 * np.max(np.abs(ob))


def test_returns_with_the_work_in_flight(kn, host, torch_cuda, monkeypatch):
    """Behind 200 ms of other work on its stream the spectrum and its gradient return at once (also in a program that
    takes the library's messages), and what follows on that stream reads finished results."""
    torch = torch_cuda
    monkeypatch.delenv("KN_VERBOSE", raising=False)
    N, nb = 64, 48
    ((F, a),) = _grids(torch, N, 1)
    on, op, _, _ = O.total_powerspectrum(F, nb)
    rc, ob = O.bin_power_adjoint(F, nb, np.ones(on))
    fn, st = knhip.power_spectrum_function(), torch.cuda.Stream()
    big = torch.empty(1 << 28, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()

    def step():
        x = a.detach().requires_grad_(True)
        p = fn.apply(x, nb)
        (bar,) = torch.autograd.grad(p.sum(), x)
        return p.detach() * 2.0, bar * 2.0

    with torch.cuda.stream(st):
        step()                      # the geometry's tables, the allocator's blocks
        torch.cuda.synchronize()
        messages = host.kn_test_messages()
        print("work in flight", flush=True)
        for _ in range(400):
            big.zero_()
        busy = torch.cuda.Event()
        busy.record()
        p, bar = step()
        assert not busy.query()
        assert host.kn_test_messages() == messages
        p, bar = p.cpu().numpy(), bar.cpu().numpy()
    np.testing.assert_allclose(p, 2.0 * op[:on], rtol=1e-12)
    e = np.max(np.abs(bar.view(np.complex128).reshape(ob.shape) - 2.0 * ob))
    assert rc == 0 and e < 1e-12 * np.max(np.abs(2.0 * ob))


def test_reports_the_mass_when_asked(kn, host, torch_cuda, monkeypatch):
    """With KN_VERBOSE set |F(0)| is reported, as total_powerspectrum does, and the spectrum is the same."""
    torch = torch_cuda
    ((F, a),) = _grids(torch, 24, 1)
    out, n = torch.zeros((2, 24), dtype=torch.float64, device="cuda"), C.c_int()
    for i in (0, 1):
        if i:
            monkeypatch.setenv("KN_VERBOSE", "1")
        else:
            monkeypatch.delenv("KN_VERBOSE", raising=False)
        before = host.kn_test_messages()
        assert kn.kn_power_spectrum_device(a.data_ptr(), 24, 24, 0, 24, out[i].data_ptr(), C.byref(n), None) == 0
        assert host.kn_test_messages() == before + i
    torch.cuda.synchronize()
    np.testing.assert_allclose(out[1].cpu().numpy(), out[0].cpu().numpy(), rtol=1e-14)
