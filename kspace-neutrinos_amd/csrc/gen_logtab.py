"""Generates kn_logtab.h: the table of the rescale sweep's log(sqrt(k2)).

P. T. P. Tang, "Table-driven implementation of the logarithm function in IEEE
floating-point arithmetic", ACM TOMS 16 (1990): the mantissa m in [1, 2) falls
in one of 128 intervals; with r_j close to 1 / (interval's centre),
log m = -log r_j + log1p(m r_j - 1), |m r_j - 1| <= 2^-8.  r_j is chosen where
-log(r_j) / 2 all but coincides with a multiple of 2^-44 (S. Gal, "Computing
elementary functions: a new approach for achieving high accuracy and good
performance", 1986): the entry then has no rounding, nor has its sum with a
binary exponent times the leading part of log(2) / 2.

    python3 gen_logtab.py > kn_logtab.h
"""
from mpmath import floor, log, mp, nint

mp.dps = 40
N = 128
UNIT = mp.mpf(2) ** -44

print("""// kn_logtab.h -- generated by gen_logtab.py; do not edit.
// kn_logtab[j] = { r_j, l_j }: r_j within 1e-10 of 1 / (1 + (j + 1/2) / 128),
// l_j = -log(r_j) / 2, a multiple of 2^-44 (to below 2^-%d).
#ifndef KN_LOGTAB_H
#define KN_LOGTAB_H

#define KN_LOGTAB_N %d
""" % (58, N))
print("static __device__ const __align__(16) double kn_logtab[2 * KN_LOGTAB_N] = {")
for j in range(N):
    r0 = mp.mpf(float(1 / (1 + (mp.mpf(j) + mp.mpf(1) / 2) / N)))
    l0, step = -log(r0) / 2 / UNIT, mp.mpf(2) ** -53
    # -log(r0 + t step) / 2 in units, to second order in t step / r0 (the third is below 1e-18 units), in 80-bit fixed point
    d, one = step / r0, 1 << 80
    c0, c1, c2 = (int(v * one) for v in (l0, d / 2 / UNIT, d * d / 4 / UNIT))
    off = lambda t: abs((c0 - t * (c1 - t * c2) + one // 2) % one - one // 2)
    best = next(t for t in range(1 << 22) if off(t) < one >> 15)
    r = r0 + best * step
    assert mp.mpf(float(r)) == r
    l = -log(r) / 2
    q = nint(l / UNIT) * UNIT
    assert mp.mpf(float(q)) == q and abs(l - q) < mp.mpf(2) ** -58
    print("    %s, %s," % (float(r).hex(), float(q).hex()))
hi = float(floor(log(2) / 2 / UNIT) * UNIT)
print("""};

// log(2) / 2 in two parts: the first has 44 binary digits, so a binary exponent times it is exact
#define KN_HALF_LN2_HI %s
#define KN_HALF_LN2_LO %s

#endif""" % (hi.hex(), float(log(2) / 2 - mp.mpf(hi)).hex()))
