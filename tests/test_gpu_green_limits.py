"""The Green's-function sweep at the largest grids it takes: one slab of a grid
whose per-axis factors fill the LDS, with and without a ratio table, to the
last size accepted, and the refusal of the next."""
import math

import numpy as np
import pytest

import knhip

pytestmark = pytest.mark.gpu

BOX = 512000.0


def _want(torch, f, N, x, y0, lk, rt, norm, asmth):
    """The two factors at rows y0 .. of slab x in plain torch."""
    i = np.arange(N)
    kv = np.where(i <= N // 2, i, i - N).astype(float)
    with np.errstate(invalid="ignore"):
        w = np.where(kv == 0, 1.0, math.pi * kv / (N * np.sin(math.pi * kv / N)))
    kv, w = torch.from_numpy(kv).cuda(), torch.from_numpy(w).cuda()
    n, h = f.shape
    ky, kz = kv[y0:y0 + n, None], torch.arange(h, dtype=torch.float64, device="cuda")[None, :]
    k2 = kv[x] ** 2 + ky ** 2 + kz ** 2
    zero = k2 == 0
    k2[zero] = 1.0
    s = torch.ones_like(k2)
    if lk is not None:
        logk = torch.clamp(0.5 * torch.log(k2) + math.log(2 * math.pi / BOX), lk[0], lk[-1])
        j = torch.clamp(torch.searchsorted(lk, logk, right=True) - 1, 0, max(len(lk) - 2, 0))
        jn = torch.clamp(j + 1, max=len(lk) - 1)
        t = (logk - lk[j]) / torch.where(jn > j, lk[jn] - lk[j], torch.ones_like(logk))
        s = 1 + norm * (rt[j] + t * (rt[jn] - rt[j]))
    g = -torch.exp(-k2 * (2 * math.pi * asmth / BOX) ** 2) / k2 * (w[x] * w[y0:y0 + n, None] * w[None, :h]) ** 4
    return torch.where(zero, torch.zeros_like(f), f * s * g)


# 16 B per bin, four buckets of 4 B each, 8 B per axis index: 160 KB hold dims 20479 without bins, 20475 with one, 18439
# with 510; with bins, from 20220 (one) and 18439 (510) the logarithm's table has no room beside them
@pytest.mark.parametrize("N,nb", [(20223, 0), (20224, 0), (20479, 0), (20219, 1), (20220, 1), (20475, 1), (20399, 20),
                                  (19455, 256), (18438, 510), (18439, 510), (18435, 511)])
def test_largest_grids(kn, torch_cuda, N, nb):
    """1e-14, as the fused sweep's other tests; the exponent is below 0.3 and the ratio's slope 0.3, so that neither its
    factors' nor log k's rounding is magnified."""
    torch = torch_cuda
    print("Green sweep, one slab", N, nb, flush=True)
    x, h, asmth, norm = (0 if nb % 2 == 0 else N - 3), N // 2 + 1, 0.1 * BOX / N, 0.07
    gen = torch.Generator(device="cuda").manual_seed(N + nb)
    f = torch.view_as_complex(torch.rand((N, h, 2), dtype=torch.float64, device="cuda", generator=gen) + 0.5)
    lk = rt = None
    args = (None, None, 0)
    if nb:
        lk = torch.linspace(math.log(2 * math.pi / BOX) + 0.2, math.log(math.pi * N / BOX) - 0.1, max(nb, 2),
                            dtype=torch.float64)[:nb].cuda()
        rt = 0.5 + 0.3 * torch.sin(lk)
        args = (lk.data_ptr(), rt.data_ptr(), nb)
    d = f.clone()
    assert kn.kn_rescale_green_device(d.data_ptr(), N, x, 1, BOX, *args, norm, asmth, None) == 0
    torch.cuda.synchronize()
    worst = 0.0
    for y0 in range(0, N, 2048):
        want = _want(torch, f[y0:y0 + 2048], N, x, y0, lk, rt, norm, asmth)
        got = d[y0:y0 + 2048]
        assert torch.all((want == 0) == (got == 0))
        e = torch.nan_to_num(torch.abs(got - want) / torch.abs(want), nan=0.0)
        worst = max(worst, float(e.max()))
    print("  worst %.2e" % worst)
    assert worst < 1e-14


def test_beyond_the_limit(kn, torch_cuda):
    """One axis index more is refused."""
    torch = torch_cuda
    d = torch.zeros(16, dtype=torch.float64, device="cuda")
    for N, nb in [(20480, 0), (20476, 1), (20400, 20), (19456, 256), (18440, 510)]:
        p = (d.data_ptr(), d.data_ptr()) if nb else (None, None)
        assert kn.kn_rescale_green_device(d.data_ptr(), N, 0, 1, BOX, *p, nb, 0.1, 1.0, None) == 3004
