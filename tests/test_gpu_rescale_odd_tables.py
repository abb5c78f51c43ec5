"""Ratio tables with values that the stored slopes cannot carry: a log k that is
not finite, ratios whose difference over a bin's width overflows."""
import ctypes as C
import math

import numpy as np
import pytest

from test_gpu_binning import _rand_grid

pytestmark = pytest.mark.gpu

BOX, NORM = 512000.0, 0.3


def _factor(k2, lk, rt):
    """The sweep's rule: the segment from the bucket of log k on, then the reference's interpolation in it."""
    n, nb = len(lk), 4 * len(lk)
    with np.errstate(all="ignore"):
        kk = 0.5 * math.log(k2) + math.log(2 * math.pi / BOX)
        kk = lk[0] if kk < lk[0] else kk
        kk = lk[-1] if kk > lk[-1] else kk
        inv_bw = nb / (lk[-1] - lk[0])
        u = (kk - lk[0]) * inv_bw
        q = 0 if math.isnan(u) else int(min(max(u, 0), nb))
        edge = lk[0] + np.float64(q) / inv_bw
        lo, hi = 0, n - 1
        while hi > lo + 1:
            mid = (lo + hi) >> 1
            lo, hi = (lo, mid) if lk[mid] > edge else (mid, hi)
        while lo < n - 2 and lk[lo + 1] <= kk:
            lo += 1
        h = lk[lo + 1] - lk[lo]
        return 1 + NORM * (rt[lo] + (kk - lk[lo]) / h * (rt[lo + 1] - rt[lo]) if h > 0 else rt[lo])


BASE = np.linspace(-13.0, -4.0, 12)


def _put(a, at, v):
    a = a.copy()
    a[at] = v
    return a


RT = np.random.default_rng(4).uniform(0, 1, 12)
TABLES = {"nan log k": (_put(BASE, 5, math.nan), RT), "nan first": (_put(BASE, 0, math.nan), RT),
          "nan last": (_put(BASE, 11, math.nan), RT), "-inf first": (_put(BASE, 0, -math.inf), RT),
          "inf last": (_put(BASE, 11, math.inf), RT), "largest": (BASE, _put(RT, 4, 1.7e308)),
          "lowest": (BASE, _put(RT, 4, -1.7e308)), "inf ratio": (BASE, _put(RT, 6, math.inf)),
          "nan ratio": (BASE, _put(RT, 6, math.nan)), "close": (-8.0 + 1e-13 * np.arange(12), 1e297 * RT)}


def _nan_flag(kn, torch):
    """The flag that NaN factors raise, read and lowered again by the rescale that takes a host table."""
    fn = kn.kn_rescale_from_host_table
    dp = C.POINTER(C.c_double)
    fn.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_double, dp, dp, C.c_int, C.c_double]
    d, t = torch.ones((4, 4, 3), dtype=torch.complex128, device="cuda"), np.array([-9.0, -8.0])
    return fn(d.data_ptr(), 4, 0, 4, BOX, t.ctypes.data_as(dp), t.ctypes.data_as(dp), 2, 0.1)


@pytest.mark.parametrize("name", list(TABLES))
@pytest.mark.parametrize("N", [12, 130])
def test_odd_tables(kn, torch_cuda, name, N):
    """Finite where the rule is, and infinite or NaN where that is (1e-13: log k's rounding over a segment's width; the close
    table within its largest ratio)."""
    torch = torch_cuda
    assert _nan_flag(kn, torch) == 0
    lk, rt = TABLES[name]
    print("odd table", name, N, flush=True)
    F = _rand_grid(N, 3, 1)
    F[:] = 1.0
    d, tab = torch.from_numpy(F).cuda(), torch.from_numpy(np.concatenate([lk, rt])).cuda()
    n = len(lk)
    assert kn.kn_rescale_device(d.data_ptr(), N, 0, 1, BOX, tab.data_ptr(), tab.data_ptr() + 8 * n, n, NORM, None) == 0
    got = d.cpu().numpy().real[0]
    assert _nan_flag(kn, torch) == int(np.any(np.isnan(got)))
    want = np.ones_like(got)
    for y in range(0, N, max(1, N // 16)):
        for z in range(N // 2 + 1):
            ky = y if y <= N // 2 else y - N
            if ky or z:
                want[y, z] = _factor(ky * ky + z * z, lk, rt)
                g, w = got[y, z], want[y, z]
                if np.isfinite(w):
                    assert abs(g - w) <= 1e-13 * abs(w) or (name == "close" and abs(g) <= 1e298)
                else:
                    assert g == w or (math.isnan(g) and math.isnan(w))
