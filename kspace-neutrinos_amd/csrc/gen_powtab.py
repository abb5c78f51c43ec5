"""Generates kn_powtab.h: the tables of x^4.1811, the power in specialJ's fit.

x = 2^e m with m in [1, 2) in one of 128 intervals; with r_j = 1 / (interval's
centre) rounded to double and r = m r_j - 1, |r| <= 2^-8 (P. T. P. Tang,
"Table-driven implementation of the logarithm function in IEEE floating-point
arithmetic", ACM TOMS 16 (1990), used for the power itself),
x^p = 2^(e p) r_j^-p (1 + r)^p.  The binomial series of (1 + r)^p is cut after r^5: its
coefficients fall fast at p = 4.1811, and r^6's is -0.0071 (below 3e-17 of the value).

    python3 gen_powtab.py > kn_powtab.h
"""
from mpmath import mp

mp.dps = 40
N, E = 128, 64
P = mp.mpf(4.1811)  # the double of delta_tot_table.c:425

print("""// kn_powtab.h -- generated by gen_powtab.py; do not edit.
// kn_powtab[j] = { r_j, r_j^-p }, r_j = 1 / (1 + (j + 1/2) / 128) rounded, p = 4.1811;
// kn_powexp[e + KN_POWTAB_E] = 2^(e p).
#ifndef KN_POWTAB_H
#define KN_POWTAB_H

#define KN_POWTAB_N %d
#define KN_POWTAB_E %d
""" % (N, E))
print("static __device__ const double kn_powtab[2 * KN_POWTAB_N] = {")
for j in range(N):
    r = float(1 / (1 + (mp.mpf(j) + mp.mpf(1) / 2) / N))
    print("    %s, %s," % (r.hex(), float(mp.mpf(r) ** -P).hex()))
print("};\n\nstatic __device__ const double kn_powexp[2 * KN_POWTAB_E + 1] = {")
for e in range(-E, E + 1):
    print("    %s," % float(mp.mpf(2) ** (e * P)).hex())
print("};\n\n// (1 + r)^p = 1 + r (A1 + r (A2 + ...))")
c = mp.mpf(1)
for k in range(1, 6):
    c = c * (P - k + 1) / k
    print("#define KN_POW_A%d %s" % (k, float(c).hex()))
print("\n#endif")
