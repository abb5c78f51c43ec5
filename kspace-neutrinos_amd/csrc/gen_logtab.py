"""Generates kn_logtab.h: the table of the rescale sweep's logarithm.

P. T. P. Tang, "Table-driven implementation of the logarithm function in IEEE
floating-point arithmetic", ACM TOMS 16 (1990): the mantissa m in [1, 2) falls
in one of 128 intervals; with r_j = 1 / (interval's centre) rounded to double,
log m = -log r_j + log1p(m r_j - 1), |m r_j - 1| <= 2^-8.

    python3 gen_logtab.py > kn_logtab.h
"""
from mpmath import log, mp

mp.dps = 40
N = 128

print("""// kn_logtab.h -- generated by gen_logtab.py; do not edit.
// kn_logtab[j] = { r_j, -log r_j }, r_j = 1 / (1 + (j + 1/2) / 128) rounded.
#ifndef KN_LOGTAB_H
#define KN_LOGTAB_H

#define KN_LOGTAB_N %d
""" % N)
print("static __device__ const __align__(16) double kn_logtab[2 * KN_LOGTAB_N] = {")
for j in range(N):
    r = float(1 / (1 + (mp.mpf(j) + mp.mpf(1) / 2) / N))
    print("    %s, %s," % (r.hex(), float(-log(mp.mpf(r))).hex()))
hi = float(mp.floor(log(2) / 2 * 2 ** 44) / 2 ** 44)
print("""};

// log(2) / 2 in two parts: the first has 44 binary digits, so a binary exponent times it is exact
#define KN_HALF_LN2_HI %s
#define KN_HALF_LN2_LO %s

#endif""" % (hi.hex(), float(log(2) / 2 - mp.mpf(hi)).hex()))
