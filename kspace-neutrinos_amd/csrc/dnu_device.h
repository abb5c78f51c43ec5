// dnu_device.h -- device building blocks of the free-streaming integral (b).
//
// Included by delta_nu.hip.  The integrand, interpolants and adaptive rule
// follow delta_tot_table.c:375-611 of the reference:
//   delta_nu(k) = IC(k) + delta_nu_prefac * int_{log T0}^{log a} I_k(x) dx,
//   I_k(x) = fsl(x) / (e^x H(e^x)) * specialJ(k fsl(x) / (m/kT), qc, nufrac_low) * S_k(x),
// with fsl a natural cubic spline through 16 Na fslength values on a uniform
// log-a grid and S_k a natural cubic spline (linear for Na = 2) through the
// stored delta_tot[k][.], integrated by QUADPACK QAG with the 61-point
// Gauss-Kronrod rule (relative tolerance 1e-6, at most 200 subintervals).
// One wavefront runs one QAG: its lanes evaluate the 61 nodes of both halves
// of the bisected interval in one pass; the interval list lives in LDS.
#ifndef KN_DNU_DEVICE_H
#define KN_DNU_DEVICE_H

#include <hip/hip_runtime.h>
#include <float.h>
#include <math.h>

#include <algorithm>
#include <vector>

#include "kn_gk61.h"
#include "kn_powtab.h"

namespace kn_dnu {

constexpr int kLimit = 200;   // QAG subinterval limit (GSL_VAL)
constexpr int kHnc = 10;      // coefficients per function per H panel
static_assert(kHnc == 10, "FslIntegrandLds steps five pairs a panel");
constexpr int kHStride = 2 * kHnc;  // one panel: 1/(a^2 H) coefficients, then 1/(a H)
// A panel whose fit misses H by more than this (relative, at test points
// between the interpolation nodes) holds a jump or a kink of H: it is split
// there into two fits, kept out of line (at most kHSplitMax per table).
constexpr double kHSplitTol = 1e-12;
constexpr int kHSplitMax = 4;
// One piece of a split panel: centre and scale of its own t = (x - centre) *
// scale, then both functions' coefficients.
constexpr int kHPiece = 2 + kHStride;
// One split record: the split point, the piece left of it, the piece right of it.
constexpr int kHSplitStride = 1 + 2 * kHPiece;

__constant__ double c_xgk[31];
__constant__ double c_wgk[31];
__constant__ double c_wg[15];

// ---- H(a) factors as functions of x = ln a: Chebyshev panels of width 1/inv_w from origin x0 ----
// Each panel holds the coefficients of 1/(a^2 H) (the fslength integrand,
// delta_tot_table.c:378-383) and of 1/(a H) (the delta_nu integrand's factor,
// :492-500), so neither integrand forms an exponential: fitted in Chebyshev
// polynomials, stored as powers of the place v in [0, 1] across the panel,
// which take half the operations (the coefficients fall by a factor of a
// thousand per degree, so nothing is lost).  H may be only
// piecewise smooth (the host's neutrino density switches from its spline
// table to the non-relativistic series at a = 100 kT/m, omega_nu_single.c:
// 171-183, where H jumps by ~1e-8 relative): a panel that holds such a point
// is split there into two fits, stored after the npanel regular panels; the
// table lists the split panels' indices.  A split panel's own coefficients are
// NaN in the device's table: the regular evaluation knows one by its value and
// compares no index.
struct HTab {
    const double *coef;  // npanel * kHStride, then nsplit * kHSplitStride
    double x0, inv_w;
    int npanel, nsplit;
    int split_p[kHSplitMax];
};

// Both functions' interpolants at the kHnc Chebyshev points of [lo, hi];
// hub(a) = H(a).  Host and device (the device background's panels).
template <typename Hub>
__host__ __device__ inline void h_fit(double lo, double hi, Hub hub, double *coef)
{
    const double half = 0.5 * (hi - lo), mid = lo + half;
    double g2[kHnc], g1[kHnc];
    for (int j = 0; j < kHnc; j++) {
        const double x = mid + half * cos(M_PI * (j + 0.5) / kHnc);
        const double h = hub(exp(x));
        g2[j] = exp(-2.0 * x) / h;
        g1[j] = exp(-x) / h;
    }
    for (int k = 0; k < kHnc; k++) {
        double s2 = 0.0, s1 = 0.0;
        for (int j = 0; j < kHnc; j++) {
            const double c = cos(M_PI * k * (j + 0.5) / kHnc);
            s2 += g2[j] * c;
            s1 += g1[j] * c;
        }
        coef[k] = (k == 0 ? 1.0 : 2.0) * s2 / kHnc;
        coef[kHnc + k] = (k == 0 ? 1.0 : 2.0) * s1 / kHnc;
    }
}

// Clenshaw sum of one function's coefficients at t in [-1, 1].
template <typename P>
__host__ __device__ __forceinline__ double h_clenshaw(P c, double t)
{
    double b1 = 0.0, b2 = 0.0;
#pragma unroll
    for (int k = kHnc - 1; k >= 1; k--) {
        const double b0 = fma(2.0 * t, b1, c[k] - b2);
        b2 = b1;
        b1 = b0;
    }
    return fma(t, b1, c[0] - b2);
}

// One function of a panel at v in [0, 1]: sum_k c[k] v^k.
template <typename P>
__host__ __device__ __forceinline__ double h_horner(P c, double v)
{
    double r = c[kHnc - 1];
#pragma unroll
    for (int k = kHnc - 2; k >= 0; k--) r = fma(r, v, c[k]);
    return r;
}

// A fit's Chebyshev coefficients (t = 2 v - 1) into the panel's powers of v,
// for both functions.
__host__ __device__ inline void h_store(const double *fit, double *panel)
{
    for (int w = 0; w < 2; w++) {
        const double *c = fit + w * kHnc;
        double *pw = panel + w * kHnc;
        double a[kHnc] = {}, b[kHnc] = {};  // T_{k-1}, T_k as powers of v
        a[0] = 1.0;
        b[0] = -1.0;
        b[1] = 2.0;
        for (int i = 0; i < kHnc; i++) pw[i] = c[0] * a[i] + c[1] * b[i];
        for (int k = 2; k < kHnc; k++) {
            double prev = 0.0;  // b[i - 1]
            for (int i = 0; i < kHnc; i++) {
                const double n = 4.0 * prev - 2.0 * b[i] - a[i];
                prev = b[i];
                a[i] = b[i];
                b[i] = n;
                pw[i] += c[k] * n;
            }
        }
    }
}

// A split panel's value: the piece left or right of the split point.
template <typename P>
__host__ __device__ __forceinline__ double h_split_eval(P rec, double x, int which)
{
    P piece = rec + 1 + (x >= rec[0] ? kHPiece : 0);
    return h_clenshaw(piece + 2 + which * kHnc, (x - piece[0]) * piece[1]);
}

// The largest relative miss of the fits `coef` of [lo, hi], at the ends and
// half-way between adjacent interpolation nodes.
template <typename Hub>
__host__ __device__ inline double h_fit_err(const double *coef, double lo, double hi, Hub hub)
{
    const double half = 0.5 * (hi - lo), mid = lo + half;
    double worst = 0.0;
    for (int j = -1; j < kHnc; j++) {
        const double t = j < 0 ? -1.0 : (j == kHnc - 1 ? 1.0 : cos(M_PI * (j + 1) / kHnc));
        const double x = mid + half * t;
        const double h = hub(exp(x));
        const double e2 = fabs(h_clenshaw(coef, t) / (exp(-2.0 * x) / h) - 1.0);
        const double e1 = fabs(h_clenshaw(coef + kHnc, t) / (exp(-x) / h) - 1.0);
        worst = fmax(worst, fmax(e2, e1));
    }
    return worst;
}

// One piece [lo, hi] of a split panel into piece[kHPiece].
template <typename Hub>
__host__ __device__ inline void h_piece(double lo, double hi, Hub hub, double *piece)
{
    const double half = 0.5 * (hi - lo);
    piece[0] = lo + half;
    piece[1] = half > 0.0 ? 1.0 / half : 0.0;
    h_fit(lo, hi, hub, piece + 2);
}

// The panel [lo, hi] into panel[kHStride].  Where the fit misses H by
// more than kHSplitTol the panel is also split, into rec[kHSplitStride], at
// the point that bisection finds (the half whose own fit misses more is
// kept, until both halves fit or the bracket is a few units in the last
// place wide).  Returns the fit's miss (above kHSplitTol: rec was written).
template <typename Hub>
__host__ __device__ inline double h_panel(double lo, double hi, Hub hub, double *panel, double *rec)
{
    double tmp[kHStride];
    h_fit(lo, hi, hub, tmp);
    const double err = h_fit_err(tmp, lo, hi, hub);
    h_store(tmp, panel);
    if (err <= kHSplitTol) return err;
    double l = lo, r = hi;
    for (;;) {
        const double m = l + 0.5 * (r - l);
        if (!(m > l && m < r)) break;
        h_fit(l, m, hub, tmp);
        const double el = h_fit_err(tmp, l, m, hub);
        h_fit(m, r, hub, tmp);
        const double er = h_fit_err(tmp, m, r, hub);
        if (el <= kHSplitTol && er <= kHSplitTol) {
            l = r = m;
            break;
        }
        if (el >= er) r = m;
        else l = m;
    }
    const double xs = l + 0.5 * (r - l);
    rec[0] = xs;
    h_piece(lo, xs, hub, rec + 1);
    h_piece(xs, hi, hub, rec + 1 + kHPiece);
    return err;
}

// Host: split records of one table, at most kHSplitMax, the panels whose
// fit misses most kept (the others keep their one-piece fit).
struct HSplits {
    int n = 0;
    int p[kHSplitMax];
    double err[kHSplitMax];
    double rec[kHSplitMax][kHSplitStride];
    // offers panel q's record; returns whether it was kept
    bool offer(int q, double e, const double *r)
    {
        int slot = n;
        if (n == kHSplitMax) {
            slot = 0;
            for (int i = 1; i < n; i++)
                if (err[i] < err[slot]) slot = i;
            if (err[slot] >= e) return false;
        } else {
            n++;
        }
        p[slot] = q;
        err[slot] = e;
        for (int i = 0; i < kHSplitStride; i++) rec[slot][i] = r[i];
        return true;
    }
};

// Host: the whole table of npanel panels of width w from x0, then the split
// records; H.split_p and H.nsplit from them.
template <typename Hub>
inline void h_table(double x0, double w, int npanel, Hub hub, std::vector<double> &coef, HTab &H)
{
    coef.assign((size_t)npanel * kHStride, 0.0);
    HSplits sp;
    double rec[kHSplitStride];
    for (int p = 0; p < npanel; p++) {
        const double e = h_panel(x0 + p * w, x0 + (p + 1) * w, hub, &coef[(size_t)p * kHStride], rec);
        if (e > kHSplitTol) sp.offer(p, e, rec);
    }
    for (int i = 0; i < sp.n; i++) {
        std::fill_n(coef.begin() + (size_t)sp.p[i] * kHStride, kHStride, NAN);
        coef.insert(coef.end(), sp.rec[i], sp.rec[i] + kHSplitStride);
    }
    H.x0 = x0;
    H.inv_w = 1.0 / w;
    H.npanel = npanel;
    H.nsplit = sp.n;
    for (int i = 0; i < kHSplitMax; i++) H.split_p[i] = i < sp.n ? sp.p[i] : -1;
}

// Device form: the table lives in global memory, so its loads are global
// loads even where the pointer came from a descriptor in memory.  A lane in
// a split panel (known by the NaN of its own coefficients) takes the
// out-of-line pieces.
typedef const __attribute__((address_space(1))) double gconst_double;

// A pointer kept in a descriptor in memory, known to point to global memory: as
// a generic one it would be used by flat accesses, which wait for the LDS
// counter too and cannot be told apart while in flight.
template <class T>
struct GlobalPtr {
    __attribute__((address_space(1))) T *p;
    __host__ __device__ __forceinline__ GlobalPtr &operator=(T *q)
    {
        p = (__attribute__((address_space(1))) T *)q;
        return *this;
    }
    __host__ __device__ __forceinline__ operator T *() const { return (T *)p; }
};

// x's panel p (clamped to the table) and the place v in [0, 1] across it.
struct HLoc {
    int p;
    double v;
};
__device__ __forceinline__ HLoc h_locate(const HTab &H, double x, int first, int last)
{
    const double u = (x - H.x0) * H.inv_w;
    HLoc L;
    L.p = (int)u;
    L.p = L.p < first ? first : (L.p > last ? last : L.p);
    L.v = u - L.p;
    return L;
}
__device__ __forceinline__ HLoc h_locate(const HTab &H, double x) { return h_locate(H, x, 0, H.npanel - 1); }

// Panel p's value at x from its split record; NaN when it has none.
__device__ __forceinline__ double h_split(const HTab &H, int p, double x, int which)
{
    int s = -1;
#pragma unroll
    for (int i = 0; i < kHSplitMax; i++)  // constant indices: the list stays in registers
        if (i < H.nsplit && p == H.split_p[i]) s = i;
    if (s >= 0)
        return h_split_eval((gconst_double *)(H.coef + (size_t)H.npanel * kHStride + (size_t)s * kHSplitStride), x,
                            which);
    return NAN;
}

// One function (which = 0: 1/(a^2 H), 1: 1/(a H)) at x; regular: NaN in a split panel.
__device__ __forceinline__ double h_regular(const HTab &H, const HLoc &L, int which)
{
    return h_horner((gconst_double *)H.coef + (unsigned)(L.p * kHStride + which * kHnc), L.v);
}
__device__ __forceinline__ double h_eval(const HTab &H, double x, int which)
{
    const HLoc L = h_locate(H, x);
    const double r = h_regular(H, L, which);
    return r == r ? r : h_split(H, L.p, x, which);
}

__device__ __forceinline__ double inv_a2h(const HTab &H, double x) { return h_eval(H, x, 0); }
__device__ __forceinline__ double inv_ah(const HTab &H, double x) { return h_eval(H, x, 1); }

// ---- the background: Omega_nu(a) and H(a), host and device ----
// The neutrino density of omega_nu_single.c:55-205 (a table of kRhoTab log-a
// points per distinct mass, each a Fermi-Dirac energy integral, interpolated
// by a natural cubic spline; the relativistic and non-relativistic limits
// outside it) and the Hubble function of the N-body code's hook (gadget-2
// patch 0003:38-55, with the kspace neutrinos and, optionally, photons).
constexpr int kRhoTab = 200;     // omega_nu_single.c:14
constexpr double kNuSw = 100.0;  // omega_nu_single.h: the series holds for kT/(a m) < 1/100
constexpr int kNuSpecies = 3;

struct BgDev {
    double Omega0, OmegaLambda, Hubble;  // Hubble: H0 in internal time units
    double rhocrit, kBtnu;               // g cm^-3 (h included); eV
    double conv;                         // (eV/c)^4 -> g cm^-3 for one species (omega_nu_single.c:100-114)
    double og;                           // Omega_g at a = 1 (omega_nu_single.c:77-81)
    double onu1;                         // Omega_nu(1)
    int radiation;                       // add Omega_g(a) (INCLUDE_RADIATION)
    int deg[kNuSpecies];                 // equal masses folded into the first (init_omega_nu)
    int tab[kNuSpecies];                 // 1: species i has a density table
    double mnu[kNuSpecies];
    const double *loga[kNuSpecies], *rho[kNuSpecies], *c2[kNuSpecies];  // kRhoTab each
};

// omega_nu_single.c:89-96: the integrand of rho_nu_init, q^2 eps(q) f0(q).
struct FdEnergy {
    double am, kT;
    __host__ __device__ double operator()(double q) const
    {
        const double eps = sqrt(q * q + am * am);
        const double f0 = 1. / (exp(q / kT) + 1);
        return q * q * eps * f0;
    }
};

// omega_nu_single.c:156-160: heavily non-relativistic, zeta(3), zeta(5) and
// zeta(7) terms.
__host__ __device__ inline double bg_nonrel(double a, double kT, double am, double r2, double conv)
{
    return am * (kT * kT * kT) / (a * a * a * a) *
           (1.5 * 1.202056903159594 + r2 * 45. / 4. * 1.0369277551433704 + 2835. / 32. * r2 * r2 * 1.0083492773819229 +
            80325 / 32. * r2 * r2 * r2 * 1.0020083928260826) *
           conv;
}

// omega_nu_single.c:164-167: heavily relativistic.
__host__ __device__ inline double bg_rel(double a, double kT, double conv)
{
    return 7 * pow(M_PI * kT / a, 4) / 120. * conv;
}

// Natural cubic spline at v (knots x, values y, second-derivative halves c;
// the interval by bisection, as gsl_interp_eval's cspline).
__host__ __device__ inline double bg_spline(const double *x, const double *y, const double *c, int n, double v)
{
    int lo = 0, hi = n - 1;
    while (hi > lo + 1) {
        const int mid = (hi + lo) / 2;
        if (x[mid] > v) hi = mid;
        else lo = mid;
    }
    const double h = x[lo + 1] - x[lo], dy = y[lo + 1] - y[lo], dx = v - x[lo];
    const double b = (dy / h) - h * (c[lo + 1] + 2.0 * c[lo]) / 3.0;
    const double d = (c[lo + 1] - c[lo]) / (3.0 * h);
    return y[lo] + dx * (b + dx * (c[lo] + dx * d));
}

// Natural cubic spline coefficients c[n] of (x, y): the tridiagonal system of
// the interior second derivatives by forward elimination and back
// substitution; work holds 3 (n - 2) doubles.
__host__ __device__ inline void bg_spline_init(const double *x, const double *y, int n, double *c, double *work)
{
    const int m = n - 2;
    for (int i = 0; i < n; i++) c[i] = 0.0;
    if (m <= 0) return;
    double *gam = work, *alp = work + m, *z = work + 2 * m;
    for (int i = 0; i < m; i++) {
        const double hl = x[i + 1] - x[i], hr = x[i + 2] - x[i + 1];
        const double gl = hl != 0.0 ? 1.0 / hl : 0.0, gr = hr != 0.0 ? 1.0 / hr : 0.0;
        const double diag = 2.0 * (hr + hl);
        const double rhs = 3.0 * ((y[i + 2] - y[i + 1]) * gr - (y[i + 1] - y[i]) * gl);
        if (m == 1) {
            c[1] = rhs / diag;
            return;
        }
        alp[i] = i == 0 ? diag : diag - (x[i + 1] - x[i]) * gam[i - 1];
        if (i < m - 1) gam[i] = hr / alp[i];
        z[i] = i == 0 ? rhs : rhs - gam[i - 1] * z[i - 1];
    }
    for (int i = 0; i < m; i++) z[i] = z[i] / alp[i];
    c[m] = z[m - 1];
    for (int i = m - 2; i >= 0; i--) c[i + 1] = z[i] - gam[i] * c[i + 2];
}

// omega_nu_single.c:171-205: the physical density of species s at a.
__host__ __device__ inline double bg_rho_nu(const BgDev &b, int s, double a)
{
    const double kT = b.kBtnu, am = a * b.mnu[s];
    const double r2 = kT * kT / am / am;
    if (kNuSw * kNuSw * r2 < 1) return bg_nonrel(a, kT, am, r2, b.conv);
    if (am < 1e-6 * kT) return bg_rel(a, kT, b.conv);
    const double la = log(a);
    if (!b.tab[s] || la < b.loga[s][0])
        return am < 1e-4 * kT ? bg_rel(a, kT, b.conv) : bg_nonrel(a, kT, am, r2, b.conv);
    return bg_spline(b.loga[s], b.rho[s], b.c2[s], kRhoTab, la);
}

// omega_nu_single.c:55-67 (get_omega_nu).
__host__ __device__ inline double bg_omega_nu(const BgDev &b, double a)
{
    double rho = 0;
    for (int i = 0; i < kNuSpecies; i++)
        if (b.deg[i] > 0) rho += b.deg[i] * bg_rho_nu(b, i, a);
    return rho / b.rhocrit;
}

// gadget-2 patch 0003:38-55: matter + Lambda + curvature, the neutrinos as
// Omega_nu(a) in place of their share of Omega0/a^3, photons when enabled.
__host__ __device__ inline double bg_hubble(const BgDev &b, double a)
{
    double omega_tot = b.Omega0 / pow(a, 3) + b.OmegaLambda + (1. - b.OmegaLambda - b.Omega0) / (a * a);
    omega_tot += bg_omega_nu(b, a) - b.onu1 / pow(a, 3);
    if (b.radiation) omega_tot += b.og / pow(a, 4);
    return b.Hubble * sqrt(omega_tot);
}

struct BgHub {
    BgDev b;
    __host__ __device__ double operator()(double a) const { return bg_hubble(b, a); }
};

// ---- the split search of h_panel by one wavefront (device-built tables) ----
// Two intervals' fits at once: lanes 0-19 sample H at the two intervals'
// kHnc interpolation nodes while lanes 20-41 sample it at their 11 check
// points (those of h_fit_err); lanes 0-39 then form one coefficient each
// (interval, function, k) and lanes 20-41 the fits' misses.  Every lane gets
// both intervals' largest misses (el, er; with check only).
struct HFit2Lds {
    double g[2][2][kHnc];  // samples: interval, function (1/(a^2 H), 1/(a H)), node
    double c[2][2][kHnc];  // coefficients
    double e[2][kHnc + 1];  // misses at the check points
};

template <typename Hub>
__device__ void h_fit2_wave(double lo0, double hi0, double lo1, double hi1, const Hub &hub, HFit2Lds &L, bool check,
                            double &el, double &er)
{
    const int lane = threadIdx.x & 63;
    double f2 = 0.0, f1 = 0.0, t = 0.0;
    if (lane < 2 * kHnc || (check && lane < 2 * kHnc + 2 * (kHnc + 1))) {
        const int iv = lane < 2 * kHnc ? lane / kHnc : (lane - 2 * kHnc) / (kHnc + 1);
        const double lo = iv ? lo1 : lo0, hi = iv ? hi1 : hi0;
        const double half = 0.5 * (hi - lo), mid = lo + half;
        if (lane < 2 * kHnc) {
            t = cos(M_PI * (lane % kHnc + 0.5) / kHnc);
        } else {
            const int j = (lane - 2 * kHnc) % (kHnc + 1) - 1;
            t = j < 0 ? -1.0 : (j == kHnc - 1 ? 1.0 : cos(M_PI * (j + 1) / kHnc));
        }
        const double x = mid + half * t;
        const double h = hub(exp(x));
        f2 = exp(-2.0 * x) / h;
        f1 = exp(-x) / h;
        if (lane < 2 * kHnc) {
            L.g[iv][0][lane % kHnc] = f2;
            L.g[iv][1][lane % kHnc] = f1;
        }
    }
    __builtin_amdgcn_wave_barrier();
    if (lane < 4 * kHnc) {
        const int iv = lane / (2 * kHnc), fn = (lane / kHnc) & 1, k = lane % kHnc;
        double s = 0.0;
        for (int j = 0; j < kHnc; j++) s += L.g[iv][fn][j] * cos(M_PI * k * (j + 0.5) / kHnc);
        L.c[iv][fn][k] = (k == 0 ? 1.0 : 2.0) * s / kHnc;
    }
    __builtin_amdgcn_wave_barrier();
    if (!check) return;
    if (lane >= 2 * kHnc && lane < 2 * kHnc + 2 * (kHnc + 1)) {
        const int iv = (lane - 2 * kHnc) / (kHnc + 1), jj = (lane - 2 * kHnc) % (kHnc + 1);
        const double e2 = fabs(h_clenshaw(L.c[iv][0], t) / f2 - 1.0);
        const double e1 = fabs(h_clenshaw(L.c[iv][1], t) / f1 - 1.0);
        L.e[iv][jj] = fmax(e2, e1);
    }
    __builtin_amdgcn_wave_barrier();
    el = 0.0;
    er = 0.0;
    for (int j = 0; j <= kHnc; j++) {
        el = fmax(el, L.e[0][j]);
        er = fmax(er, L.e[1][j]);
    }
    __builtin_amdgcn_wave_barrier();
}

// h_panel's split of [lo, hi] (bisection until both halves fit, then both
// pieces' fits) by one wavefront into rec[kHSplitStride].  Every lane keeps
// the same bracket, so the loop ends together.
template <typename Hub>
__device__ void h_split_wave(double lo, double hi, const Hub &hub, double *rec, HFit2Lds &L)
{
    double l = lo, r = hi, el, er;
    for (;;) {
        const double m = l + 0.5 * (r - l);
        if (!(m > l && m < r)) break;
        h_fit2_wave(l, m, m, r, hub, L, true, el, er);
        if (el <= kHSplitTol && er <= kHSplitTol) {
            l = r = m;
            break;
        }
        if (el >= er) r = m;
        else l = m;
    }
    const double xs = l + 0.5 * (r - l);
    h_fit2_wave(lo, xs, xs, hi, hub, L, false, el, er);
    const int lane = threadIdx.x & 63;
    if (lane < 2 * kHStride) {
        const int iv = lane / kHStride, i = lane % kHStride;
        rec[1 + iv * kHPiece + 2 + i] = L.c[iv][i / kHnc][i % kHnc];
    } else if (lane < 2 * kHStride + 2) {
        const int iv = lane - 2 * kHStride;
        const double plo = iv ? xs : lo, phi = iv ? hi : xs, half = 0.5 * (phi - plo);
        rec[1 + iv * kHPiece] = plo + half;
        rec[1 + iv * kHPiece + 1] = half > 0.0 ? 1.0 / half : 0.0;
    } else if (lane == 2 * kHStride + 2) {
        rec[0] = xs;
    }
    __builtin_amdgcn_wave_barrier();
}

// 1/d from the hardware estimate refined by one Newton step (relative error
// a few units in the last place, against ten instructions for a division);
// d finite and normal.
__device__ __forceinline__ double rcp_fast(double d)
{
    const double r = __builtin_amdgcn_rcp(d);
    return fma(r, fma(-d, r, 1.0), r);
}

// ---- special functions (delta_tot_table.c:417-463) ----
struct JPar {
    double qc, nufrac_low;
    double en[20];  // exp(-n qc) for n = 1..19, from the host
};

__device__ __forceinline__ double sph_j0(double x)
{
    if (fabs(x) < 0.5) {
        const double y = x * x;
        return 1.0 + y * (-1.0 / 6.0 + y * (1.0 / 120.0 + y * (-1.0 / 5040.0 + y * (1.0 / 362880.0 +
                         y * (-1.0 / 39916800.0 + y * (1.0 / 6227020800.0))))));
    }
    return sin(x) / x;
}

// The hybrid series of specialJ (delta_tot_table.c:435-463),
//   sum_{n=1}^{19} (-1)^{n+1} e^{-n qc} [A_n qc j0 + B_n cos(qc x)] / (n^2 + x^2)^2,
//   A_n = n^2 + n^3 qc + n qc x^2 - x^2,  B_n = 2n + n^2 qc + qc x^2,
// with each bracket regrouped by powers of n,
//   A_n qc j0 + B_n c = n^2 al + n^3 be + n ga + de,
//   al = qc j0 + qc c, be = qc^2 j0, ga = qc^2 x^2 j0 + 2c, de = qc x^2 c - qc x^2 j0,
// so that a term is three fused multiply-adds, the squared denominator's
// reciprocal and one more fused multiply-add.  SJTerms holds one point's
// per-x factors; specialJ and specialJ2 run the same operations per point, four
// terms at a time: their weights come by one scalar load (757 k x 2000 steps:
// 103 us, with two at a time 108, with all nineteen 130 for the registers).
struct SJTerms {
    double y, al, be, ga, de, integ;
};
__device__ __forceinline__ SJTerms sj_terms(double x, double qc)
{
    double s, c;
    sincos(qc * x, &s, &c);
    const double j0 = fabs(qc * x) < 0.5 ? sph_j0(qc * x) : s / (qc * x);
    const double y = x * x, qj = qc * j0;
    return {y, qj + qc * c, qc * qj, qc * (y * qj) + 2.0 * c, qc * y * c - y * qj, 0.0};
}
__device__ __forceinline__ void sj_term(SJTerms &t, int n, double w)
{
    const double fn = (double)n, n2 = fn * fn, n3 = n2 * fn;
    const double ii = fma(n2, t.al, fma(n3, t.be, fma(fn, t.ga, t.de)));
    const double d = n2 + t.y;
    t.integ = fma(w * rcp_fast(d * d), ii, t.integ);
}
// x^4.1811 of the fit, x > 0, within 2 units in the last place (kn_powtab.h:
// two table entries and five terms) where exp(4.1811 log x), with the
// product's rounding in the exponent, was off by up to 30, for a quarter of the
// operations.  Outside 2^-64 .. 2^64, where the fit's other terms leave nothing of
// it, and for infinities and NaN, which they carry, any finite value does (not
// so for the derivative's x^4.1811 / x below 2^-64: specialJ_d leaves it out).
// QAG of 256 histories 455 -> 438 us, of 12 histories of 16-96 k 22.8 -> 18.2.
__device__ __forceinline__ double pow_fit(double x)
{
    long long u;
    __builtin_memcpy(&u, &x, sizeof u);
    const int hi = (int)(u >> 32), e0 = (hi >> 20) - 1023, j = (hi >> 13) & (KN_POWTAB_N - 1);
    const int e = e0 < -KN_POWTAB_E ? -KN_POWTAB_E : (e0 > KN_POWTAB_E ? KN_POWTAB_E : e0);
    const long long mu = (u & 0xfffffffffffffLL) | 0x3ff0000000000000LL;
    double m;
    __builtin_memcpy(&m, &mu, sizeof m);
    const double t = kn_powtab[2 * j + 1], r = fma(m, kn_powtab[2 * j], -1.0);
    const double q = r * fma(r, fma(r, fma(r, fma(r, KN_POW_A5, KN_POW_A4), KN_POW_A3), KN_POW_A2), KN_POW_A1);
    return kn_powexp[e + KN_POWTAB_E] * fma(t, q, t);
}

__device__ __forceinline__ double sj_fit(double x0)
{
    const double x = x0 <= 0. ? 1. : x0;  // a select, not a branch: two points' chains then overlap
    const double x2 = x * x, x4 = x2 * x2, x8 = x4 * x4;
    const double v = (1. + 0.0168 * x2 + 0.0407 * x4) / (1. + 2.1734 * x2 + 1.6787 * pow_fit(x) + 0.1467 * x8);
    return x0 <= 0. ? 1. : v;
}

// HYB false: every species of the launch has qc = 0, and the series is left out
// (its registers, and the sine's, would be held through the fit's code too).
template <bool HYB = true>
__device__ __forceinline__ double specialJ(double x, const JPar &P)
{
    if (HYB && P.qc > 0) {
        SJTerms t = sj_terms(x, P.qc);
#pragma unroll 4
        for (int n = 1; n < 20; n++) sj_term(t, n, ((n & 1) ? 1.0 : -1.0) * P.en[n]);
        return t.integ / (1.5 * 1.202056903159594 * (1 - P.nufrac_low));
    }
    return sj_fit(x);
}

// specialJ at two points, the two series in one loop (two independent
// chains per term); each point's operations are specialJ's.
template <bool HYB>
__device__ __forceinline__ void specialJ2(double x1, double x2, const JPar &P, double &j1, double &j2)
{
    if (HYB && P.qc > 0) {
        SJTerms t1 = sj_terms(x1, P.qc), t2 = sj_terms(x2, P.qc);
#pragma unroll 4
        for (int n = 1; n < 20; n++) {
            const double w = ((n & 1) ? 1.0 : -1.0) * P.en[n];
            sj_term(t1, n, w);
            sj_term(t2, n, w);
        }
        j1 = t1.integ / (1.5 * 1.202056903159594 * (1 - P.nufrac_low));
        j2 = t2.integ / (1.5 * 1.202056903159594 * (1 - P.nufrac_low));
        return;
    }
    j1 = sj_fit(x1);
    j2 = sj_fit(x2);
}

// ---- natural cubic spline evaluation, GSL cspline/linear semantics ----
__device__ __forceinline__ double cspline_val(double xl, double xr, double yl, double yr, double ci, double ci1,
                                              double x)
{
    const double h = xr - xl, ih = rcp_fast(h);
    const double dy = yr - yl;
    const double dx = x - xl;
    const double b = dy * ih - h * (ci1 + 2.0 * ci) * (1.0 / 3.0);
    const double d = (ci1 - ci) * ih * (1.0 / 3.0);
    return yl + dx * (b + dx * (ci + dx * d));
}

__device__ __forceinline__ double linear_val(double xl, double xr, double yl, double yr, double x)
{
    const double h = xr - xl;
    if (h > 0.0) return yl + (x - xl) / h * (yr - yl);
    return yl;
}

// The fslength table's knots are x0 + i (xa - x0) / (n - 1.) (delta_tot_table.c:582),
// the expression the fslength kernels store them with: knot i recomputed here
// equals the stored one, so the spline is evaluated without loading knots.
// The quotient is formed from 1 / den, rounded, and one correction by its
// exact remainder (Markstein 1990), which gives the division's own result in a
// quarter of its instructions.
struct UniformKnots {
    double x0, span, den, rden;  // x0, xa - x0, n - 1., 1 / (n - 1.)
    __device__ __forceinline__ double at(int i) const
    {
        const double p = i * span, q = p * rden;
        return x0 + fma(fma(-q, den, p), rden, q);
    }
};

// settle() on those knots: i and its interval [xl, xr]
__device__ __forceinline__ int settle_uniform(const UniformKnots &u, int n, int i, double x, double &xl, double &xr)
{
    i = i < 0 ? 0 : (i > n - 2 ? n - 2 : i);
    xl = u.at(i);
    while (i > 0 && xl > x) xl = u.at(--i);
    xr = u.at(i + 1);
    while (i < n - 2 && xr <= x) {
        xl = xr;
        xr = u.at(++i + 1);
    }
    return i;
}

// One step of settle_uniform either way from the guess, without its loops: the
// rounding of (x - x0) / h moves the guess by one knot at most unless the knots
// are a few units in the last place apart.  settled: whether x's interval was
// reached, i.e. settle_uniform's answer.
__device__ __forceinline__ int step_uniform(const UniformKnots &u, int n, int i, double x, double &xl, double &xr,
                                            bool &settled)
{
    i = i < 0 ? 0 : (i > n - 2 ? n - 2 : i);
    const double l = u.at(i), r = u.at(i + 1);
    i += (int)(i < n - 2 && r <= x) - (int)(i > 0 && l > x);
    xl = u.at(i);
    xr = u.at(i + 1);
    settled = !(i > 0 && xl > x) && !(i < n - 2 && xr <= x);
    return i;
}

// Largest i <= n-2 with xa[i] <= x, starting from a guess (GSL bsearch result).
__device__ __forceinline__ int settle(const double *xa, int n, int i, double x)
{
    i = i < 0 ? 0 : (i > n - 2 ? n - 2 : i);
    while (i > 0 && xa[i] > x) i--;
    while (i < n - 2 && xa[i + 1] <= x) i++;
    return i;
}

// ---- integrands ----
struct FslIntegrand {  // delta_tot_table.c:378-383: 1 / a / (a H(a))
    HTab H;
    // NaN in a split panel, and the value there
    __device__ __forceinline__ double regular(double x) const { return h_regular(H, h_locate(H, x), 0); }
    __device__ __forceinline__ double split(double x) const { return h_split(H, h_locate(H, x).p, x, 0); }
    __device__ __forceinline__ double operator()(double x) const { return inv_a2h(H, x); }
};

// The same with the 1/(a^2 H) coefficients of panels p0 .. p1 in LDS, kHnc
// doubles a panel.  The points' panels lie among them, but for a point that its
// rounding carries past the last: it takes the last panel's fit, as beyond a table.
struct alignas(16) HPair {
    double x, y;
};
struct FslIntegrandLds {
    HTab H;
    const HPair *c;  // 16-byte aligned: a pair is one LDS read, whose passes of 16 lanes take one or two panels each
    int p0, p1;
    __device__ __forceinline__ double regular(double x) const
    {
        const HLoc L = h_locate(H, x, p0, p1);
        const int i0 = L.p - p0;
        const HPair *q = c + (i0 + (i0 << 2));  // kHnc / 2 pairs a panel (shifts: a 32-bit multiply takes four times as long)
        HPair k = q[kHnc / 2 - 1];
        double r = fma(k.y, L.v, k.x);
#pragma unroll
        for (int i = kHnc / 2 - 2; i >= 0; i--) {
            k = q[i];
            r = fma(fma(r, L.v, k.y), L.v, k.x);
        }
        return r;
    }
    __device__ __forceinline__ double split(double x) const { return h_split(H, h_locate(H, x, p0, p1).p, x, 0); }
};

template <bool HYB>
struct DnuIntegrand {  // delta_tot_table.c:492-500
    HTab H;
    const double *fy, *fc;  // fslength spline on the uniform knots fk
    UniformKnots fk;
    int nfs;
    double fx0, fxhi, finv_h;    // first and last knot, 1 / spacing
    const double *sx, *sy, *sc;  // delta_tot spline of this k
    const int *sbucket;
    int ns, nsb, linear;
    double sx0, sxhi, sinv_bw;   // first and last stored step
    double k, mnubykT, k_by_m;  // k_by_m = k / mnubykT
    const JPar *J;  // in device memory: the series weights are read where used
    int *edom;
    // One point's place in the tables: its knot intervals, the fslength spline's values and 1 / (a H).
    struct Point {
        bool in;
        int si;
        double xl, xr, f0, f1, g0, g1;  // fslength: interval, values, coefficients
        double sl, sr;                  // delta_tot's interval
        double ih;
    };
    // Straight-line code, so that the loads of both points are in flight together:
    // one step from the fslength guess, the bucket's knot or one of the next two.
    // again: x lies further off (walk() finds it).
    __device__ __forceinline__ Point place(double x, bool &again) const
    {
        Point p;
        p.in = !(x < fx0 || x > fxhi || x < sx0 || x > sxhi);
        int q = (int)((x - sx0) * sinv_bw);
        q = q < 0 ? 0 : (q > nsb ? nsb : q);
        const int b = sbucket[q];
        bool settled;
        const int fi = step_uniform(fk, nfs, (int)((x - fx0) * finv_h), x, p.xl, p.xr, settled);
        p.f0 = fy[fi], p.f1 = fy[fi + 1], p.g0 = fc[fi], p.g1 = fc[fi + 1];
        const HLoc L = h_locate(H, x);
        p.ih = h_regular(H, L, 1);
        const int i = b < 0 ? 0 : (b > ns - 2 ? ns - 2 : b), last = ns - 1;
        const int i1 = i + 1, i2 = i + 2 < last ? i + 2 : last, i3 = i + 3 < last ? i + 3 : last;
        const double t0 = sx[i], t1 = sx[i1], t2 = sx[i2], t3 = sx[i3];
        const bool up1 = i1 < last && t1 <= x, up2 = i2 < last && t2 <= x, up3 = i3 < last && t3 <= x;
        p.si = up1 ? (up2 ? i2 : i1) : i;
        p.sl = up1 ? (up2 ? t2 : t1) : t0;
        p.sr = up1 ? (up2 ? t3 : t2) : t1;
        again = !settled || (i > 0 && t0 > x) || up3 || p.ih != p.ih;
        return p;
    }
    // The same from any distance, and in a split H panel.
    __device__ __forceinline__ void walk(double x, Point &p) const
    {
        const int fi = settle_uniform(fk, nfs, (int)((x - fx0) * finv_h), x, p.xl, p.xr);
        p.f0 = fy[fi], p.f1 = fy[fi + 1], p.g0 = fc[fi], p.g1 = fc[fi + 1];
        p.si = settle(sx, ns, p.si, x);
        p.sl = sx[p.si], p.sr = sx[p.si + 1];
        if (p.ih != p.ih) p.ih = h_split(H, h_locate(H, x).p, x, 1);
    }
    // Two points.  A used point outside the tables flags GSL_EDOM and gives 0;
    // the indices of every point are clamped into the tables, so an unused or
    // outside point reads in bounds.  (With the knot walks as loops, a branch per
    // spline interval and the series' code beside the fit's, a rule took 9000-11000
    // clocks.)
    __device__ __forceinline__ void eval2(double x1, double x2, bool use1, bool use2, double &r1, double &r2) const
    {
        bool again1, again2;
        Point p1 = place(x1, again1), p2 = place(x2, again2);
        if (again1) walk(x1, p1);
        if (again2) walk(x2, p2);
        const double y10 = sy[p1.si], y11 = sy[p1.si + 1], c10 = sc[p1.si], c11 = sc[p1.si + 1];
        const double y20 = sy[p2.si], y21 = sy[p2.si + 1], c20 = sc[p2.si], c21 = sc[p2.si + 1];
        const double fsl1 = cspline_val(p1.xl, p1.xr, p1.f0, p1.f1, p1.g0, p1.g1, x1);
        const double fsl2 = cspline_val(p2.xl, p2.xr, p2.f0, p2.f1, p2.g0, p2.g1, x2);
        double j1, j2, dt1, dt2;
        specialJ2<HYB>(k_by_m * fsl1, k_by_m * fsl2, *J, j1, j2);
        if (linear) {
            dt1 = linear_val(p1.sl, p1.sr, y10, y11, x1);
            dt2 = linear_val(p2.sl, p2.sr, y20, y21, x2);
        } else {
            dt1 = cspline_val(p1.sl, p1.sr, y10, y11, c10, c11, x1);
            dt2 = cspline_val(p2.sl, p2.sr, y20, y21, c20, c21, x2);
        }
        r1 = p1.in ? fsl1 * p1.ih * j1 * dt1 : 0.0;  // fsl / (a H) specJ dtot
        r2 = p2.in ? fsl2 * p2.ih * j2 * dt2 : 0.0;
        if ((use1 && !p1.in) || (use2 && !p2.in)) atomicOr(edom, 1);  // GSL_EDOM in gsl_interp_eval -> terminate(2001)
    }
};

// The integrand at two points of one lane: f.eval2 where the integrand has
// it, else two calls.
template <class F>
__device__ __forceinline__ void eval_pair(const F &f, double x1, double x2, bool use1, bool use2, double &r1,
                                          double &r2)
{
    r1 = use1 ? f(x1) : 0.0;
    r2 = use2 ? f(x2) : 0.0;
}
template <bool HYB>
__device__ __forceinline__ void eval_pair(const DnuIntegrand<HYB> &f, double x1, double x2, bool use1, bool use2,
                                          double &r1, double &r2)
{
    f.eval2(x1, x2, use1, use2, r1, r2);
    r1 = use1 ? r1 : 0.0;
    r2 = use2 ? r2 : 0.0;
}

// ---- moves between lanes ----
// A wavefront that runs one QAG spends its time in a serial chain: a rule's
// four sums of five steps each were most of it while every step went through
// the LDS crossbar (over 100 clocks).  These run in the vector unit (8 to 16).
// All 64 lanes take part.  (The host build of this file, a test's emulation,
// has the shuffles.)
#if defined(__HIP_DEVICE_COMPILE__)
template <int CTRL>
__device__ __forceinline__ int dpp(int v)
{
    return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);  // a lane without a source keeps its own
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v)
{
    return __hiloint2double(dpp<CTRL>(__double2hiint(v)), dpp<CTRL>(__double2loint(v)));
}
// v of the next lane (lane 63: its own), of the one before (lane 0: its own)
template <class T>
__device__ __forceinline__ T lane_next(T v)
{
    return dpp<0x130>(v);  // wave_shl:1
}
template <class T>
__device__ __forceinline__ T lane_prev(T v)
{
    return dpp<0x138>(v);  // wave_shr:1
}
__device__ __forceinline__ double lane_value(double v, int l)  // l the same in all lanes
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

// The sum over each 32-lane half in every lane, by the butterfly v += v[lane ^
// m], m = 16, 8, 4, 2, 1 (a step's two orders of its pair give one sum).
__device__ __forceinline__ double half_sum(double v)
{
    // rows 0 and 1 (2 and 3) of 16 lanes: the swap leaves one row's values in both rows, the other's likewise
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
    v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    v += dpp<0x128>(v);  // row_ror:8
    v += dpp<0x124>(v);  // row_ror:4, lane ^ 4's value now that lane ^ 8 holds the same
    v += dpp<0x4e>(v);   // quad_perm [2,3,0,1]
    v += dpp<0xb1>(v);   // quad_perm [1,0,3,2]
    return v;
}
#else
template <class T>
__device__ __forceinline__ T lane_next(T v)
{
    const int p = threadIdx.x & 63;
    return __shfl(v, p < 63 ? p + 1 : 63, 64);
}
template <class T>
__device__ __forceinline__ T lane_prev(T v)
{
    const int p = threadIdx.x & 63;
    return __shfl(v, p > 0 ? p - 1 : 0, 64);
}
__device__ __forceinline__ double lane_value(double v, int l)
{
    return __shfl(v, l, 64);
}
__device__ __forceinline__ double half_sum(double v)
{
    for (int m = 16; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}
#endif

// t^1.5 rounded once: t sqrt(t) carried in two parts (the products' and the
// square root's rounding errors recovered exactly by fma), then summed.  The
// plain t * sqrt(t) rounds twice and differs from the correctly rounded
// value in about a quarter of all t, which could reorder QUADPACK's error
// list against a libm pow(t, 1.5).
__device__ __forceinline__ double pow_three_halves(double t)
{
#pragma clang fp contract(off)  // p must be the rounded product for e to be its error
    const double s = sqrt(t);
    const double r = fma(-s, s, t);  // t - s^2, exact
    const double p = t * s;
    const double e = fma(t, s, -p);  // t s - p, exact
    return p + (e + t * r / (2 * s));
}

__device__ __forceinline__ double gk_rescale(double err, double resabs, double resasc)
{
    err = fabs(err);
    if (resasc != 0 && err != 0) {
        // QUADPACK's rescale: resasc min(1, (200 err / resasc)^1.5)
        const double t = 200 * err / resasc;
        const double s = pow_three_halves(t);
        err = s < 1 ? resasc * s : resasc;
    }
    if (resabs > DBL_MIN / (50 * DBL_EPSILON)) {
        const double floor_err = 50 * DBL_EPSILON * resabs;
        if (floor_err > err) err = floor_err;
    }
    return err;
}

struct GK {
    double res, err, resabs, resasc;
};

// The rule's node and weights of a lane of gk61_pair, read once per QAG.
struct RuleLane {
    double x, wk, wg;
    __device__ __forceinline__ RuleLane()
    {
        const int j = threadIdx.x & 31;
        x = j <= 30 ? c_xgk[j] : 0.0;
        wk = j <= 30 ? c_wgk[j] : 0.0;
        wg = (j < 30 && (j & 1)) ? c_wg[j >> 1] : 0.0;
    }
};

// 61-point Gauss-Kronrod on [a1,b1] (lanes 0-31) and [a2,b2] (lanes 32-63).
template <class F>
__device__ __forceinline__ void gk61_pair(const F &f, const RuleLane &rule, double a1, double b1, double a2, double b2,
                                          GK &g1, GK &g2)
{
#pragma clang fp contract(off)  // every product and sum rounded as written (gk61_first's sums match bit for bit)
    const int lane = threadIdx.x & 63, hf = lane >> 5, j = lane & 31;
    const double a = hf ? a2 : a1, b = hf ? b2 : b1;
    const double c = 0.5 * (a + b), h = 0.5 * (b - a);
    // lane 30 takes the centre (c_xgk[30] = 0: c - 0 is c) in the same
    // evaluation as the other lanes' left nodes, so a wavefront runs the
    // integrand twice, not three times
    double f1 = 0.0, f2 = 0.0;
    {
        const double dx = j <= 30 ? h * rule.x : 0.0;
        eval_pair(f, c - dx, c + dx, j <= 30, j < 30, f1, f2);
    }
    const double wk = rule.wk, wgv = rule.wg;
    const double sk = half_sum(j == 30 ? wk * f1 : wk * (f1 + f2));
    const double sg = half_sum(wgv * (f1 + f2));
    const double sa = half_sum(j == 30 ? wk * fabs(f1) : wk * (fabs(f1) + fabs(f2)));
    const double mean = sk * 0.5;
    const double sasc = half_sum(j == 30 ? wk * fabs(f1 - mean) : (j < 30 ? wk * (fabs(f1 - mean) + fabs(f2 - mean)) : 0.0));
    GK r;
    r.res = sk * h;
    r.resabs = sa * fabs(h);
    r.resasc = sasc * fabs(h);
    r.err = gk_rescale((sk - sg) * h, r.resabs, r.resasc);
    // broadcast each half's result to every lane
    g1.res = lane_value(r.res, 0);
    g1.err = lane_value(r.err, 0);
    g1.resabs = lane_value(r.resabs, 0);
    g1.resasc = lane_value(r.resasc, 0);
    g2.res = lane_value(r.res, 32);
    g2.err = lane_value(r.err, 32);
    g2.resabs = lane_value(r.resabs, 32);
    g2.resasc = lane_value(r.resasc, 32);
}

// The rule's nodes and weights by gk61_pair's lane j (0 at j = 31, and Gauss
// weights at even j), from constant memory or from a copy in LDS: with j
// different from lane to lane, constant memory means vector loads.
struct RuleConst {
    __device__ __forceinline__ double x(int j) const { return j <= 30 ? c_xgk[j] : 0.0; }
    __device__ __forceinline__ double wk(int j) const { return j <= 30 ? c_wgk[j] : 0.0; }
    __device__ __forceinline__ double wg(int j) const { return (j < 30 && (j & 1)) ? c_wg[j >> 1] : 0.0; }
};
constexpr int kRuleLds = 96;  // doubles
struct RuleLds {
    const double *k;
    __device__ __forceinline__ double x(int j) const { return k[j]; }
    __device__ __forceinline__ double wk(int j) const { return k[32 + j]; }
    __device__ __forceinline__ double wg(int j) const { return k[64 + j]; }
};
// The copy, by the first 32 threads of a block.
__device__ __forceinline__ void rule_to_lds(double *k)
{
    const RuleConst c;
    const int j = threadIdx.x;
    if (j < 32) {
        k[j] = c.x(j);
        k[32 + j] = c.wk(j);
        k[64 + j] = c.wg(j);
    }
}

// QAG's first step on [a, b], a <= b, by four lanes of a
// wavefront, lanes l, l ^ 16, l ^ 32, l ^ 48 (quarter q = (l >> 4) & 3; the
// other 15 lanes of each quarter take 15 other intervals, so that lanes of
// one load instruction evaluate nearby points of nearby intervals).  Quarter
// q evaluates gk61_pair's lanes j and j + 16 for j = q, q + 4, q + 8, q + 12
// and adds their terms as gk61_pair's butterfly does (xor 16, 8 and 4 within
// the quarter), then xor 2 and xor 1 across quarters (lane xor 32, 16): the
// sums, and so the estimate, are gk61_pair's bit for bit, in all four lanes.
// Returns what wave_qag61 does with the first estimate *res at relative
// tolerance epsrel: 0 it is the result, 18 roundoff, -1 bisect (valid in
// quarter 0).
// The error estimate asks for two more sums over the points, |f| and
// |f - mean|, but most integrals are accepted without them.  With f > 0
// throughout, resabs is the result itself.  For two points of weight w, resasc
// >= h w |f1 - f2| =: s; and with e the difference of the two rules, t = 200 e
// / resasc < 1/2 gives err = max(resasc t^1.5, 50 eps resabs) <= max(200 e, 50
// eps resabs), below resasc if s > 100 eps resabs.  So 200 e < s / 2, 200 e
// below the tolerance and s above that floor mean acceptance; where that is
// not so for some lane the wavefront forms the sums.
template <class F, class K>
__device__ __forceinline__ int gk61_first(const F &f, const K &k, double a, double b, double epsrel, double *res)
{
#pragma clang fp contract(off)  // as gk61_pair
    const int q = (threadIdx.x >> 4) & 3;
    const double c = 0.5 * (a + b), h = 0.5 * (b - a);
    double f01[4], f02[4], f11[4], f12[4], tk[4], tg[4];
    // four points at a time in straight-line code (sixteen would take 478 registers)
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int j0 = q + 4 * r, j1 = j0 + 16;
        const double dx0 = h * k.x(j0), dx1 = h * k.x(j1);
        const double x01 = c - dx0, x02 = c + dx0, x11 = c - dx1, x12 = c + dx1;
        double v01 = f.regular(x01), v02 = f.regular(x02), v11 = f.regular(x11), v12 = f.regular(x12);
        const double any = (v01 + v02) + (v11 + v12);
        if (__ballot(any != any)) {  // points in split panels
            if (v01 != v01) v01 = f.split(x01);
            if (v02 != v02) v02 = f.split(x02);
            if (v11 != v11) v11 = f.split(x11);
            if (v12 != v12) v12 = f.split(x12);
        }
        f01[r] = v01;
        f02[r] = v02;
        f11[r] = j1 <= 30 ? v11 : 0.0;  // j1 = 30 is the centre, which the right point repeats; 31 (quarter 3) no point
        f12[r] = j1 < 30 ? v12 : 0.0;
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int j0 = q + 4 * r, j1 = j0 + 16;
        tk[r] = k.wk(j0) * (f01[r] + f02[r]) + k.wk(j1) * (f11[r] + f12[r]);  // the centre: f12 = 0
        tg[r] = k.wg(j0) * (f01[r] + f02[r]) + k.wg(j1) * (f11[r] + f12[r]);
    }
    double least = fmin(f01[0], f02[0]);
#pragma unroll
    for (int r = 0; r < 4; r++) {
        least = fmin(least, fmin(f01[r], f02[r]));
        if (q + 4 * r + 16 < 30) least = fmin(least, fmin(f11[r], f12[r]));
        else if (q + 4 * r + 16 == 30) least = fmin(least, f11[r]);
    }
    // xor 8 (j, j + 8: r, r + 2), xor 4 (j, j + 4: r 0, 1), then across quarters
    auto sum4 = [](const double(&t)[4]) {
        double v = (t[0] + t[2]) + (t[1] + t[3]);
        v += __shfl_xor(v, 32, 64);
        v += __shfl_xor(v, 16, 64);
        return v;
    };
    const double sk = sum4(tk), sg = sum4(tg);
    *res = sk * h;
    const double tol = epsrel * fabs(*res);
    const double e200 = 200 * fabs((sk - sg) * h), s = h * k.wk(q) * fabs(f01[0] - f02[0]);
    const bool sure = least > 0 && e200 < 0.5 * s && e200 < 0.99 * tol && s > 101 * DBL_EPSILON * *res &&
                      51 * DBL_EPSILON * *res < tol;
    if (!__ballot(a < b && !sure)) return 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int j0 = q + 4 * r, j1 = j0 + 16;
        const double wk0 = c_wgk[j0], wk1 = j1 <= 30 ? c_wgk[j1] : 0.0;
        tk[r] = wk0 * (fabs(f01[r]) + fabs(f02[r])) +
                (j1 == 30 ? wk1 * fabs(f11[r]) : wk1 * (fabs(f11[r]) + fabs(f12[r])));
    }
    const double sa = sum4(tk);
    const double mean = sk * 0.5;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int j0 = q + 4 * r, j1 = j0 + 16;
        const double wk0 = c_wgk[j0], wk1 = j1 <= 30 ? c_wgk[j1] : 0.0;
        tk[r] = wk0 * (fabs(f01[r] - mean) + fabs(f02[r] - mean)) +
                (j1 == 30 ? wk1 * fabs(f11[r] - mean)
                          : (j1 < 30 ? wk1 * (fabs(f11[r] - mean) + fabs(f12[r] - mean)) : 0.0));
    }
    const double resasc = sum4(tk) * fabs(h), resabs = sa * fabs(h);
    const double err = gk_rescale((sk - sg) * h, resabs, resasc);
    if (err <= 50 * DBL_EPSILON * resabs && err > tol) return 18;
    return ((err <= tol && err != resasc) || err == 0.0) ? 0 : -1;
}

// Interval list of one wavefront (QUADPACK workspace), in LDS.  QUADPACK's
// level counts are left out: only QAGS's extrapolation reads them.
struct QagWs {
    double lo[kLimit], hi[kLimit], r[kLimit], e[kLimit];
    int ord[kLimit];
};

// Keep ord[] partially sorted by error, as QUADPACK's dqpsrt.  All lanes run
// it on identical values.
__device__ __forceinline__ void qag_sort(QagWs &w, int n, int limit, int &nrmax, int &imax)
{
    const int last = n - 1;
    int nr = nrmax, im = w.ord[nr], top, i, k;
    if (last < 2) {
        w.ord[0] = 0;
        w.ord[1] = 1;
        imax = im;
        return;
    }
    const double emax = w.e[im];
    while (nr > 0 && emax > w.e[w.ord[nr - 1]]) {
        w.ord[nr] = w.ord[nr - 1];
        nr--;
    }
    top = last < limit / 2 + 2 ? last : limit - last + 1;
    for (i = nr + 1; i < top && emax < w.e[w.ord[i]]; i++) w.ord[i - 1] = w.ord[i];
    w.ord[i - 1] = im;
    const double emin = w.e[last];
    for (k = top - 1; k > i - 2 && emin >= w.e[w.ord[k]]; k--) w.ord[k + 1] = w.ord[k];
    w.ord[k + 1] = last;
    imax = w.ord[nr];
    nrmax = nr;
}

// qag_sort with nrmax = 0 (QAG never moves it; only QAGS's extrapolation
// does), by all 64 lanes of the wavefront: the two linear scans become
// wavefront searches for the first position where the scan would stop, and
// the shifts become parallel moves (each lane reads its entry before any
// lane writes; a wavefront's LDS accesses complete in program order).  The
// list comes out exactly as qag_sort leaves it.  Returns ord[0].
__device__ __forceinline__ int qag_sort_wave(QagWs &w, int n, int limit)
{
    const int lane = threadIdx.x & 63;
    const int last = n - 1;
    const int im = w.ord[0];
    if (last < 2) {
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) {
            w.ord[0] = 0;
            w.ord[1] = 1;
        }
        return im;
    }
    const double emax = w.e[im];
    __builtin_amdgcn_wave_barrier();  // every lane has read ord[0] before it moves
    const int top = last < limit / 2 + 2 ? last : limit - last + 1;
    // i = first p in [1, top) where !(emax < e[ord[p]]), else top
    int i = top;
    for (int p0 = 1; p0 < top; p0 += 64) {
        const int p = p0 + lane;
        const unsigned long long m = __ballot(p < top && !(emax < w.e[w.ord[p]]));
        if (m) {
            i = p0 + __ffsll((long long)m) - 1;
            break;
        }
    }
    // ord[p - 1] = ord[p] for p in [1, i), then ord[i - 1] = im
    for (int p0 = 1; p0 < i; p0 += 64) {
        const int p = p0 + lane;
        const int v = p < i ? w.ord[p] : 0;
        __builtin_amdgcn_wave_barrier();
        if (p < i) w.ord[p - 1] = v;
        __builtin_amdgcn_wave_barrier();
    }
    if (lane == 0) w.ord[i - 1] = im;
    __builtin_amdgcn_wave_barrier();
    // k = largest p in [i - 1, top - 1] where !(emin >= e[ord[p]]), else i - 2
    const double emin = w.e[last];
    int k = i - 2;
    for (int p0 = top - 1; p0 > i - 2; p0 -= 64) {
        const int p = p0 - lane;
        const unsigned long long m = __ballot(p > i - 2 && !(emin >= w.e[w.ord[p]]));
        if (m) {
            k = p0 - (__ffsll((long long)m) - 1);
            break;
        }
    }
    // ord[p + 1] = ord[p] for p in [k + 1, top - 1], then ord[k + 1] = last
    for (int p0 = top - 1; p0 > k; p0 -= 64) {
        const int p = p0 - lane;
        const int v = p > k ? w.ord[p] : 0;
        __builtin_amdgcn_wave_barrier();
        if (p > k) w.ord[p + 1] = v;
        __builtin_amdgcn_wave_barrier();
    }
    if (lane == 0) w.ord[k + 1] = last;
    __builtin_amdgcn_wave_barrier();
    return w.ord[0];
}

// The same error order held by the wavefront in registers while the list
// is short: lane p keeps ord[p] (os) and that interval's error (es).  While
// fewer than limit / 2 + 2 intervals are listed, dqpsrt's top is the last
// index, so the whole order is kept sorted; the two scans are wavefront
// searches on es and the two shifts are moves between neighbouring lanes.
// ord[0] (im) was just bisected: emax is the error of the half it kept,
// emin that of the half appended at index last.  Returns the new ord[0].
#ifndef KN_WAVE_ORD
#define KN_WAVE_ORD 64
#endif
constexpr int kWaveOrd = KN_WAVE_ORD;  // most intervals held in registers
__device__ __forceinline__ int wave_ord_insert(double &es, int &os, int im, double emax, double emin, int last)
{
    const int p = threadIdx.x & 63;
    if (last < 2) {
        es = p == 0 ? emax : emin;
        os = p;
        return 0;
    }
    const int top = last;
    // i = first p in [1, top) where !(emax < e[ord[p]]), else top
    const unsigned long long m1 = __ballot(p >= 1 && p < top && !(emax < es));
    const int i = m1 ? __ffsll((long long)m1) - 1 : top;
    // ord[p - 1] = ord[p] for p in [1, i), then ord[i - 1] = im
    const double es_dn = lane_next(es);
    const int os_dn = lane_next(os);
    if (p < i - 1) {
        es = es_dn;
        os = os_dn;
    } else if (p == i - 1) {
        es = emax;
        os = im;
    }
    // k = largest p in [i - 1, top - 1] where !(emin >= e[ord[p]]), else i - 2
    const unsigned long long m2 = __ballot(p >= i - 1 && p <= top - 1 && !(emin >= es));
    const int k = m2 ? 63 - __builtin_clzll(m2) : i - 2;
    // ord[p + 1] = ord[p] for p in [k + 1, top - 1], then ord[k + 1] = last
    const double es_up = lane_prev(es);
    const int os_up = lane_prev(os);
    if (p > k + 1 && p <= top) {
        es = es_up;
        os = os_up;
    } else if (p == k + 1) {
        es = emin;
        os = last;
    }
    return __builtin_amdgcn_readfirstlane(os);
}

// The order after appending interval n - 1: in registers while it fits,
// else (once, when it outgrows them) copied to w.ord and kept there by
// qag_sort_wave.  w holds the bisected interval's new values already.
__device__ __forceinline__ int ord_insert(QagWs &w, double &es, int &os, bool &in_lds, int im, double emax,
                                          double emin, int n, int limit)
{
    if (!in_lds && n <= kWaveOrd && n - 1 < limit / 2 + 2) return wave_ord_insert(es, os, im, emax, emin, n - 1);
    if (!in_lds) {
        const int p = threadIdx.x & 63;
        if (p < n - 1) w.ord[p] = os;
        __builtin_amdgcn_wave_barrier();
        in_lds = true;
    }
    return qag_sort_wave(w, n, limit);
}

// ord[r] (r < the interval count), from wherever the order is kept; every
// lane of the wavefront calls it.
__device__ __forceinline__ int ord_rank(const QagWs &w, int os, bool in_lds, int r)
{
    const int v = __shfl(os, r & 63, 64);
    return in_lds ? w.ord[r] : v;
}

// QAG (QUADPACK dqage semantics, GSL's qag.c control flow) by one wavefront.
// Returns 0 on success or the GSL errno (11 iteration limit, 18 roundoff,
// 21 bad integrand); *result is the sum over the final subintervals.  Every
// lane keeps the same scalar state; lane 0 alone writes the intervals, and
// all lanes keep the error order together (qag_sort_wave), whose wavefront
// operations order lane 0's writes before the other lanes' reads.
template <class F>
__device__ int wave_qag61(const F &f, double a, double b, double epsrel, int limit, QagWs &w, double *result,
                          int *nint)
{
    // the first estimate and the bisections share one copy of the rule's code
    // (the integrand inlined at two places is beyond the instruction cache)
    const bool lead = (threadIdx.x & 63) == 0;
    const RuleLane rule;
    int imax = 0, os = 0;
    bool ord_lds = false;
    double es = 0.0, tol = 0.0, area = 0.0, errsum = 0.0;  // es, os: the error order in registers (ord_insert)
    double ri = 0.0, ei = 0.0, a1 = a, b1 = b, a2 = a, b2 = b;
    int n = 0, it = 1, rt1 = 0, rt2 = 0, etype = 0;
    for (;;) {
        GK g1, g2;
        gk61_pair(f, rule, a1, b1, a2, b2, g1, g2);
        if (n == 0) {
            *result = g1.res;
            *nint = 1;
            if (lead) {
                w.lo[0] = a;
                w.hi[0] = b;
                w.r[0] = g1.res;
                w.e[0] = g1.err;
                w.ord[0] = 0;
            }
            imax = __shfl(0, 0, 64);
            es = g1.err;
            tol = epsrel * fabs(g1.res);
            if (g1.err <= 50 * DBL_EPSILON * g1.resabs && g1.err > tol) return 18;
            if ((g1.err <= tol && g1.err != g1.resasc) || g1.err == 0.0) return 0;
            if (limit == 1) return 11;
            area = g1.res;
            errsum = g1.err;
            n = 1;
        } else {
            const int im = imax;
            const double r12 = g1.res + g2.res, e12 = g1.err + g2.err;
            errsum += e12 - ei;
            area += r12 - ri;
            if (g1.resasc != g1.err && g2.resasc != g2.err) {
                if (fabs(ri - r12) <= 1.0e-5 * fabs(r12) && e12 >= 0.99 * ei) rt1++;
                if (it >= 10 && e12 > ei) rt2++;
            }
            tol = epsrel * fabs(area);
            if (errsum > tol) {
                const double t = (1 + 100 * DBL_EPSILON) * (fabs(a2) + 1000 * DBL_MIN);
                if (rt1 >= 6 || rt2 >= 20) etype = 2;
                if (fabs(a1) <= t && fabs(b2) <= t) etype = 3;
            }
            if (lead) {
                if (g2.err > g1.err) {
                    w.lo[im] = a2;
                    w.r[im] = g2.res;
                    w.e[im] = g2.err;
                    w.lo[n] = a1;
                    w.hi[n] = b1;
                    w.r[n] = g1.res;
                    w.e[n] = g1.err;
                } else {
                    w.hi[im] = b1;
                    w.r[im] = g1.res;
                    w.e[im] = g1.err;
                    w.lo[n] = a2;
                    w.hi[n] = b2;
                    w.r[n] = g2.res;
                    w.e[n] = g2.err;
                }
            }
            const bool hi2 = g2.err > g1.err;
            imax = ord_insert(w, es, os, ord_lds, im, hi2 ? g2.err : g1.err, hi2 ? g1.err : g2.err, n + 1, limit);
            n++;
            it++;
            if (!(it < limit && !etype && errsum > tol)) break;
        }
        const double ai = w.lo[imax], bi = w.hi[imax];
        ri = w.r[imax];
        ei = w.e[imax];
        a1 = ai;
        b1 = a2 = 0.5 * (ai + bi);
        b2 = bi;
    }
    double s = 0.0;
    for (int k = 0; k < n; k++) s += w.r[k];
    *result = s;
    *nint = n;
    if (errsum <= tol) return 0;
    if (etype == 2) return 18;
    if (etype == 3) return 21;
    if (it == limit) return 11;
    return 5;
}

// ---- QAG by W wavefronts with speculative bisections ----
// wave_qag61's algorithm on one block of W wavefronts.  The chain of
// bisections is serial (each choice waits for the previous estimates), so
// the other wavefronts evaluate ahead: every pass each wavefront evaluates
// the two halves of one interval -- the interval to bisect now, then the two
// halves it will be cut into (one of them is next when the cut leaves it the
// largest error, as in the long chains of oscillatory integrands), then the
// next interval(s) in QUADPACK's error order (ord[]) -- and wavefront 0 runs
// wave_qag61's update for as long as the interval to bisect next has its
// halves evaluated (an interval is known by its bounds: the list holds
// disjoint intervals).  The evaluations are gk61_pair's and the update is
// wave_qag61's, so the decisions and results are wave_qag61's bit for bit;
// an evaluation that the update does not reach is only work lost.
// Estimated errors of the intervals the bisection now in hand will create,
// as fractions of its error, when they compete for a slot with the next
// intervals in error order.  The chains of the oscillatory hybrid integrand
// alternate between the next interval in order and a half of the one just
// bisected, mostly the right half, sometimes twice running.
constexpr double kRightErr = 0.1, kLeftErr = 0.05, kRightRightErr = 0.05;
struct QagSlot {
    int used, eval;    // holds an interval; evaluate it this pass
    double lo, hi;     // the interval
    GK g1, g2;         // its halves
};

template <int W>
struct QagBlock {
    QagWs ws;
    QagSlot slot[W];
    int rc, n;         // return code (-1: running) and interval count, from wavefront 0
};

template <int W, class F>
__device__ int block_qag61(const F &f, double a, double b, double epsrel, int limit, QagBlock<W> &S, double *result,
                           int *nint)
{
    const int wave = threadIdx.x >> 6;
    const bool lead = threadIdx.x == 0;  // lane 0 of wavefront 0 writes the list and the slots
    QagWs &w = S.ws;
    // pass 0: wavefront 0 the first estimate; wavefront 1 the halves of [a, b] (the first bisection)
    const RuleLane rule;
    GK g0, gx;
    if (wave <= 1) {
        const double m = 0.5 * (a + b);
        gk61_pair(f, rule, a, wave ? m : b, wave ? m : a, b, g0, gx);
        if (wave == 1 && (threadIdx.x & 63) == 0) {
            S.slot[1].used = 1;
            S.slot[1].lo = a;
            S.slot[1].hi = b;
            S.slot[1].g1 = g0;
            S.slot[1].g2 = gx;
        }
    }
    if (lead)
        for (int q = 0; q < W; q++)
            if (q != 1) S.slot[q].used = 0;
    __syncthreads();
    // wavefront 0's scalar state (identical in its 64 lanes)
    double area = 0.0, errsum = 0.0, tol = 0.0;
    int n = 1, it = 1, rt1 = 0, rt2 = 0, etype = 0, imax = 0, rc = -1;
    double es = g0.err;  // the error order in registers (ord_insert)
    int os = 0;
    bool ord_lds = false;
    if (wave == 0) {
        if (lead) {
            w.lo[0] = a;
            w.hi[0] = b;
            w.r[0] = g0.res;
            w.e[0] = g0.err;
            w.ord[0] = 0;
            }
        tol = epsrel * fabs(g0.res);
        if (g0.err <= 50 * DBL_EPSILON * g0.resabs && g0.err > tol) rc = 18;
        else if ((g0.err <= tol && g0.err != g0.resasc) || g0.err == 0.0) rc = 0;
        else if (limit == 1) rc = 11;
        area = g0.res;
        errsum = g0.err;
        imax = __shfl(0, 0, 64);
    }
    for (;;) {
        if (wave == 0) {
            // the bisections whose halves are at hand, exactly as wave_qag61's loop
            double pa = 0.0, pb = 0.0, pe = 0.0;  // the last interval looked at: the next to bisect
            while (rc < 0) {
                const int im = imax;
                const double ai = w.lo[im], bi = w.hi[im], ri = w.r[im], ei = w.e[im];
                pa = ai, pb = bi, pe = ei;
                int s = -1;
#pragma unroll
                for (int q = 0; q < W; q++)
                    if (S.slot[q].used && S.slot[q].lo == ai && S.slot[q].hi == bi) s = q;
                // every lane has read the interval before lane 0 rewrites it below
                __builtin_amdgcn_wave_barrier();
                if (s < 0) break;
                const double a1 = ai, b1 = 0.5 * (ai + bi), a2 = b1, b2 = bi;
                const GK g1 = S.slot[s].g1, g2 = S.slot[s].g2;
                const double r12 = g1.res + g2.res, e12 = g1.err + g2.err;
                errsum += e12 - ei;
                area += r12 - ri;
                if (g1.resasc != g1.err && g2.resasc != g2.err) {
                    if (fabs(ri - r12) <= 1.0e-5 * fabs(r12) && e12 >= 0.99 * ei) rt1++;
                    if (it >= 10 && e12 > ei) rt2++;
                }
                tol = epsrel * fabs(area);
                if (errsum > tol) {
                    const double t = (1 + 100 * DBL_EPSILON) * (fabs(a2) + 1000 * DBL_MIN);
                    if (rt1 >= 6 || rt2 >= 20) etype = 2;
                    if (fabs(a1) <= t && fabs(b2) <= t) etype = 3;
                }
                if (lead) {
                            if (g2.err > g1.err) {
                        w.lo[im] = a2;
                        w.r[im] = g2.res;
                        w.e[im] = g2.err;
                        w.lo[n] = a1;
                        w.hi[n] = b1;
                        w.r[n] = g1.res;
                        w.e[n] = g1.err;
                    } else {
                        w.hi[im] = b1;
                        w.r[im] = g1.res;
                        w.e[im] = g1.err;
                        w.lo[n] = a2;
                        w.hi[n] = b2;
                        w.r[n] = g2.res;
                        w.e[n] = g2.err;
                    }
                }
                const bool hi2 = g2.err > g1.err;
                imax = ord_insert(w, es, os, ord_lds, im, hi2 ? g2.err : g1.err, hi2 ? g1.err : g2.err, n + 1, limit);
                n++;
                it++;
                if (!(it < limit && !etype && errsum > tol)) {
                    rc = errsum <= tol ? 0 : etype == 2 ? 18 : etype == 3 ? 21 : it == limit ? 11 : 5;
                }
            }
            // the next pass's intervals: slot 0 the one to bisect now (never
            // evaluated yet: it would have been used above); slots 1.. the
            // W - 1 largest by error of the next W - 1 intervals in error
            // order, the two halves of the one bisected now and its right
            // half's right half, the new intervals' errors estimated as
            // fractions of its error.  An interval a slot already holds stays
            // there unevaluated; a slot not chosen keeps what it holds (the
            // list only ever splits its intervals, so a held interval is
            // either still listed with those halves or gone).
            // Lane c of wavefront 0 weighs candidate c.
            if (lead) {
                S.rc = rc;
                S.n = n;
            }
            if (rc < 0) {  // wavefront 0's state: uniform
                const int lane = threadIdx.x & 63;
                const double lo = pa, hi = pb, m = 0.5 * (lo + hi), e0 = pe;  // w's values at imax
                // the extra candidates, in lane order W - 1.. and by estimated
                // error: the right half, the left half, the right half's right half
                const double eR = kRightErr * e0, eL = kLeftErr * e0, eRR = kRightRightErr * e0;
                double cl = 0.0, ch = 0.0, ce = 0.0;
                bool has = false;
                const int ri = ord_rank(w, os, ord_lds, lane + 1 < n ? lane + 1 : 0);
                if (lane < W - 1) {
                    if (lane + 1 < n) {
                        const int i = ri;
                        cl = w.lo[i];
                        ch = w.hi[i];
                        ce = w.e[i];
                        has = true;
                    }
                } else if (lane == W - 1) {
                    cl = m, ch = hi, ce = eR, has = true;
                } else if (lane == W) {
                    cl = lo, ch = m, ce = eL, has = true;
                } else if (lane == W + 1) {
                    cl = 0.5 * (m + hi), ch = hi, ce = eRR, has = true;
                }
                // rank by error among the candidates, the lower lane first on
                // ties: the intervals in error order come sorted and so do the
                // extras, so an extra's rank counts the intervals at or above
                // its error, and an interval's the extras above its error
                const bool ordc = lane < W - 1 && has;
                const int nR = __popcll(__ballot(ordc && ce >= eR)), nL = __popcll(__ballot(ordc && ce >= eL));
                const int nRR = __popcll(__ballot(ordc && ce >= eRR));
                const int rank = lane < W - 1 ? lane + (eR > ce) + (eL > ce) + (eRR > ce)
                                 : lane == W - 1 ? nR
                                 : lane == W     ? nL + 1
                                                 : nRR + 2;
                const bool take = has && rank < W - 1;
                int held = 0;  // the slot (1..) that already holds this candidate
#pragma unroll
                for (int q = 1; q < W; q++)
                    if (S.slot[q].used && S.slot[q].lo == cl && S.slot[q].hi == ch) held = q;
                const bool keep = take && held > 0, place = take && held == 0;
                unsigned kept = 0;  // bit q: slot q keeps a chosen interval
#pragma unroll
                for (int q = 1; q < W; q++)
                    if (__ballot(keep && held == q)) kept |= 1u << q;
                const unsigned long long pl = __ballot(place);
                // the j-th candidate to place (in lane order) goes to the j-th slot not kept
                const int j = __popcll(pl & ((1ull << lane) - 1));
                int slot = 0, free = 0;
#pragma unroll
                for (int q = 1; q < W; q++)
                    if (!(kept >> q & 1)) {
                        if (free == j) slot = q;
                        free++;
                    }
                unsigned fresh = 0;
#pragma unroll
                for (int q = 1; q < W; q++)
                    if (__ballot(place && slot == q)) fresh |= 1u << q;
                __builtin_amdgcn_wave_barrier();  // every lane has read the slots before any lane writes
                if (place && slot > 0) {
                    QagSlot &sl = S.slot[slot];
                    sl.used = 1;
                    sl.lo = cl;
                    sl.hi = ch;
                }
                if (lane == 0) {
                    S.slot[0].used = 1;
                    S.slot[0].lo = lo;
                    S.slot[0].hi = hi;
                    S.slot[0].eval = 1;
                } else if (lane < W) {
                    S.slot[lane].eval = (int)(fresh >> lane & 1);
                }
            }
        }
        __syncthreads();
        if (S.rc >= 0) break;
        {
            QagSlot &sl = S.slot[wave];
            if (sl.eval) {
                const double lo = sl.lo, hi = sl.hi, m = 0.5 * (lo + hi);
                GK g1, g2;
                gk61_pair(f, rule, lo, m, m, hi, g1, g2);
                if ((threadIdx.x & 63) == 0) {
                    sl.g1 = g1;
                    sl.g2 = g2;
                }
            }
        }
        __syncthreads();
    }
    const int nn = S.n;
    double s = 0.0;
    for (int k = 0; k < nn; k++) s += w.r[k];
    *result = s;
    *nint = nn;
    return S.rc;
}

// ---- natural cubic spline coefficients, windowed parallel solve ----
// The interior system h_{i-1} c_{i-1} + 2(h_{i-1}+h_i) c_i + h_i c_{i+1} = g_i is
// 2:1 diagonally dominant, so the influence of a row decays as 0.268^distance
// on even knots and faster than 0.5^distance on any.  A window solves rows
// [lo-halo, hi+halo) with zero boundary values at the window edges and keeps
// rows [lo, hi): the edge error reaching the kept rows is 0.268^48 ~ 1e-27
// relative on even knots, below 0.5^48 ~ 4e-15 on any.
constexpr int kHalo = 48;

// ---- natural-spline rows by wavefront scans -------------------------------
// One wavefront solves a window of up to 64 kRun interior rows of
// M c = rhs (rows i = 1..n-2, c_0 = c_{n-1} = 0), lane l taking kRun
// consecutive rows in registers, and keeps the rows [lo, hi) that lie kHalo
// rows or more inside the window (zero values are assumed just outside it).
// M's L D L^T factors
//   alp_i = 2(hl_i + hr_i) - hl_i gam_{i-1},  gam_i = hr_i / alp_i
// are those of the elimination from row 1; the gam recurrence contracts by
// at most (hl/alp)(hr/alp) <= 1/4 per row, so a lane that starts it kWarm
// rows before its run (alp = diagonal there) reaches them to below
// 0.25^32 ~ 5e-20 relative.  The forward substitution
// z_i = rhs_i - gam_{i-1} z_{i-1} and the back substitution
// c_i = z_i / alp_i - gam_i c_{i+1} are first-order linear recurrences: each
// lane composes its run into one affine map, a 64-lane scan of the maps
// gives every lane its incoming value, and the lane replays its run.
constexpr int kWarm = 32;
constexpr int kRun = 10;                        // rows per lane
constexpr int kKeep = 64 * kRun - 2 * kHalo;    // rows kept per window (544)

// A lane's share of a window: rows [s, s + len) of the window's interior
// rows [wa, wb).
struct TriLane {
    int wa, wb, s, len;
};

__device__ __forceinline__ TriLane tri_lane(int n, int lo, int hi)
{
    const int lane = threadIdx.x & 63;
    TriLane t;
    t.wa = lo - kHalo;
    t.wb = hi + kHalo;  // window of interior rows [wa, wb)
    if (t.wa < 1) t.wa = 1;
    if (t.wb > n - 1) t.wb = n - 1;
    t.s = t.wa + lane * kRun;
    t.len = t.s < t.wb ? (t.wb - t.s < kRun ? t.wb - t.s : kRun) : 0;
    return t;
}

// The lane's factors gam (g) and 1 / alp (ial) over its run, and gam_{s-1} (0
// before the window's first row); past the run both are 0, so that the solve
// gives 0 there.
__device__ __forceinline__ void tri_factor(const double *x, const TriLane &t, double (&g)[kRun], double (&ial)[kRun],
                                           double &g_before)
{
    const int s = t.s, wb = t.wb, len = t.len;
    int a = s - kWarm;
    if (a < 1) a = 1;
    double gp = 0.0;
    for (int r = a; r < s && r < wb; r++) {
        const double hl = x[r] - x[r - 1], hr = x[r + 1] - x[r];
        const double diag = 2.0 * (hr + hl);
        const double alr = r == a ? diag : diag - hl * gp;
        gp = hr / alr;
    }
    g_before = s == t.wa ? 0.0 : gp;
#pragma unroll
    for (int j = 0; j < kRun; j++) {
        double gj = 0.0, aj = 0.0;
        if (j < len) {
            const int i = s + j;
            const double hl = x[i] - x[i - 1], hr = x[i + 1] - x[i];
            const double diag = 2.0 * (hr + hl);
            const double al = i == a ? diag : diag - hl * gp;
            gp = gj = hr / al;
            aj = 1.0 / al;
        }
        g[j] = gj;
        ial[j] = aj;
    }
}

// What the substitutions' scans over the lanes multiply by, from the factors
// alone: a lane's run composes to z_out = A - f[0] z_in (A from the row's
// values), and f[k] is the factor of the 2^k runs that end with the lane's;
// b[k] likewise backwards.  Three levels reach 8 runs, 80 rows: each row passes
// on at most gam of what reaches it, 0.268 on even knots (1e-46 over 80 rows),
// below 1/2 on any (alp_i > 2 hr_i + 1.5 hl_i): 0.5^80 = 8e-25, and to come near
// that every interval has to be many times the one before it.  (All six levels:
// the coefficient rows of 256 histories took 754 us for 721.)
constexpr int kScan = 3;
static_assert((kRun << kScan) >= kHalo, "the scans reach as far as a window's halo");
struct TriScan {
    double f[kScan], b[kScan];
};

__device__ __forceinline__ TriScan tri_scan(const double (&g)[kRun], double g_before)
{
    const int lane = threadIdx.x & 63;
    TriScan S;
    double f = -g_before, b = 1.0;
#pragma unroll
    for (int j = 1; j < kRun; j++) f = -g[j - 1] * f;
#pragma unroll
    for (int j = kRun - 1; j >= 0; j--) b = -g[j] * b;
#pragma unroll
    for (int k = 0; k < kScan; k++) {
        S.f[k] = f;
        S.b[k] = b;
        const double fp = __shfl_up(f, 1 << k, 64), bn = __shfl_down(b, 1 << k, 64);
        f = lane >= (1 << k) ? f * fp : f;
        b = lane + (1 << k) < 64 ? b * bn : b;
    }
    return S;
}

// Called by all 64 lanes of a wavefront together, with hi - lo <= kKeep and
// n >= 3, given the lane's factors and their scan products.
// ADJ_RHS: instead of storing the solution z, add its image under the
// transpose of the natural-spline right-hand side's y-derivative onto out
// (the second half of the spline adjoint) for the kept rows, with the
// reciprocal knot spacings ih.
// OUT: where the kept rows go (set for the solution, add for ADJ_RHS); IH:
// the reciprocal spacings.  Each kept row receives exactly one set or add.
template <class RHS, bool ADJ_RHS, class OUT, class IH>
__device__ __forceinline__ void tri_solve(int n, const RHS &rhs, int lo, int hi, const OUT &out, const TriLane &t,
                                          const double (&g)[kRun], const double (&ial)[kRun], double g_before,
                                          const TriScan &S, const IH &ih)
{
    const int lane = threadIdx.x & 63;
    const int wb = t.wb, s = t.s, len = t.len;
    double zz[kRun];
#pragma unroll
    for (int j = 0; j < kRun; j++) zz[j] = j < len ? rhs(s + j) : 0.0;
    // forward: z_i = rhs_i - gam_{i-1} z_{i-1}, z_{wa-1} = 0
    double A = zz[0];
#pragma unroll
    for (int j = 1; j < kRun; j++) A = zz[j] - g[j - 1] * A;
#pragma unroll
    for (int k = 0; k < kScan; k++) {
        const double Ap = __shfl_up(A, 1 << k, 64);
        if (lane >= (1 << k)) A = A + S.f[k] * Ap;
    }
    double z = __shfl_up(A, 1, 64);
    if (lane == 0) z = 0.0;
#pragma unroll
    for (int j = 0; j < kRun; j++) {
        z = zz[j] - (j == 0 ? g_before : g[j - 1]) * z;
        zz[j] = z * ial[j];
    }
    // back: c_i = zz_i - gam_i c_{i+1}, c_{wb} = 0
    A = 0.0;
#pragma unroll
    for (int j = kRun - 1; j >= 0; j--) A = zz[j] - g[j] * A;
#pragma unroll
    for (int k = 0; k < kScan; k++) {
        const double An = __shfl_down(A, 1 << k, 64);
        if (lane + (1 << k) < 64) A = A + S.b[k] * An;
    }
    double c = __shfl_down(A, 1, 64);
    if (lane == 63) c = 0.0;
    if (!ADJ_RHS) {
#pragma unroll
        for (int j = kRun - 1; j >= 0; j--) {
            const int i = s + j;
            c = zz[j] - g[j] * c;
            if (j < len && i >= lo && i < hi) out.set(i, c);
        }
        if (lane == 0) {
            if (lo == 0) out.set(0, 0.0);
            if (lo <= n - 1 && n - 1 < hi) out.set(n - 1, 0.0);
        }
        return;
    }
    // ADJ_RHS: out (+)= d(rhs)/dy^T z for the kept rows, with
    // rhs_i = 3 ((y_{i+1} - y_i) / h_i - (y_i - y_{i-1}) / h_{i-1}) and z_0 = z_{n-1} = 0
    double zv[kRun];
#pragma unroll
    for (int j = kRun - 1; j >= 0; j--) zv[j] = c = zz[j] - g[j] * c;
    // z just before and after this lane's run (0 at the natural ends; a
    // window's inner ends are never next to a kept row)
    double zp = __shfl_up(zv[kRun - 1], 1, 64), zn = __shfl_down(zv[0], 1, 64);
    if (lane == 0 || s - 1 < 1) zp = 0.0;
    if (lane == 63 || s + len >= wb) zn = 0.0;
#pragma unroll
    for (int j = 0; j < kRun; j++) {
        const int i = s + j;
        if (j < len && i >= lo && i < hi) {
            const double zl = j > 0 ? zv[j - 1] : zp, zr = j + 1 < len ? zv[j + 1] : zn;
            const double wl = 3.0 * ih(i - 1), wr = 3.0 * ih(i);
            double acc = 0.0;
            if (i - 1 >= 1) acc += zl * wl;
            acc -= zv[j] * (wr + wl);
            if (i + 1 <= n - 2) acc += zr * wr;
            out.add(i, acc);
        }
    }
    if (lane == 0 && lo == 0 && len > 0) out.add(0, zv[0] * (3.0 * ih(0)));  // row 0: the z_1 term
    if (lo <= n - 1 && n - 1 < hi) {                                         // row n-1: the z_{n-2} term
#pragma unroll
        for (int j = 0; j < kRun; j++)
            if (j < len && s + j == n - 2) out.add(n - 1, zv[j] * (3.0 * ih(n - 2)));
    }
}

// The windows of rows that share their knots: one for up to 64 kRun interior
// rows, else equal shares of at most kKeep kept rows (window w keeps
// [w keep, (w + 1) keep)).
__host__ __device__ inline int fac_windows(int n) { return n <= 64 * kRun + 2 ? 1 : (n + kKeep - 1) / kKeep; }
__host__ __device__ inline int fac_keep(int n)
{
    const int w = fac_windows(n);
    return (n + w - 1) / w;
}

// Factors of the knots x[0..n) stored once for every row that shares them:
// window w at fac + w kFacStride, [j][lane] for gam, then 1 / alp, then
// gam_{s-1} per lane (from the values tri_factor forms in each wavefront).
constexpr int kFacStride = (2 * kRun + 1) * 64;

__device__ __forceinline__ void tri_factor_store(const double *x, int n, int w, double *fac)
{
    const int lane = threadIdx.x & 63;
    const int keep = fac_keep(n), lo = w * keep, hi = lo + keep < n ? lo + keep : n;
    const TriLane t = tri_lane(n, lo, hi);
    double g[kRun], ial[kRun], gb;
    tri_factor(x, t, g, ial, gb);
    double *f = fac + (size_t)w * kFacStride;
#pragma unroll
    for (int j = 0; j < kRun; j++) {
        f[j * 64 + lane] = g[j];
        f[(kRun + j) * 64 + lane] = ial[j];
    }
    f[2 * kRun * 64 + lane] = gb;
}

// The span of a window in LDS: its rows and their two neighbours.
constexpr int kTriSpan = 64 * kRun + 2;
constexpr int kTriPass = (kTriSpan + 63) / 64;  // 64-wide passes over a span

// A wavefront's LDS writes ordered before its lanes' reads of them (LDS
// operations of one wavefront complete in order; the fences keep the
// compiler from moving accesses across).
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// v = src[0 .. cnt), cnt <= kTriSpan, spread over the 64 lanes: every load
// issued at once.
__device__ __forceinline__ void load_span(double (&v)[kTriPass], const double *__restrict__ src, int cnt)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int p = 0; p < kTriPass; p++) {
        const int k = p * 64 + lane;
        v[p] = k < cnt ? src[k] : 0.0;
    }
}

__device__ __forceinline__ void store_span(double *dst, const double (&v)[kTriPass], int cnt)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int p = 0; p < kTriPass; p++) {
        const int k = p * 64 + lane;
        if (k < cnt) dst[k] = v[p];
    }
}

// Right-hand side of the natural-spline system (GSL cspline): 3 (dy/h right -
// dy/h left), from staged y and ih (ys[k] = y[base + k]).
struct SplineRhsLds {
    const double *ys, *ihs;
    int base;
    __device__ __forceinline__ double operator()(int i) const
    {
        const int k = i - base;
        return 3.0 * ((ys[k + 1] - ys[k]) * ihs[k] - (ys[k] - ys[k - 1]) * ihs[k - 1]);
    }
};
struct OutLds {  // kept row i at o[i - lo]
    double *o;
    int lo;
    __device__ __forceinline__ void set(int i, double v) const { o[i - lo] = v; }
    __device__ __forceinline__ void add(int i, double v) const { o[i - lo] += v; }
};
struct IhLds {
    const double *ihs;
    int base;
    __device__ __forceinline__ double operator()(int i) const { return ihs[i - base]; }
};
struct RunRhs {  // the lane's own rows, in registers
    const double (&v)[kRun];
    int s;
    __device__ __forceinline__ double operator()(int i) const { return v[i - s]; }
};

// The lane's stored factors of window w.
__device__ __forceinline__ void tri_factor_load(const double *__restrict__ fac, int w, double (&g)[kRun],
                                                double (&ial)[kRun], double &gb)
{
    const int lane = threadIdx.x & 63;
    const double *f = fac + (size_t)w * kFacStride;
#pragma unroll
    for (int j = 0; j < kRun; j++) {
        g[j] = f[j * 64 + lane];
        ial[j] = f[(kRun + j) * 64 + lane];
    }
    gb = f[2 * kRun * 64 + lane];
}

// Spline coefficients for window w of a wavefront's rows r0, r0 + step, ... <
// rend, on knots whose factors are stored (fac_windows(n) windows, then the
// reciprocal spacings): the coefficients of row Y + r ystride go to C + r
// ystride.  The window is staged through LDS (sa: kTriSpan doubles of the
// wavefront's own; sb: the reciprocal spacings, the same for the block's
// wavefronts, which come here together): lane l solves rows s .. s + kRun - 1,
// kRun rows from its neighbours', so read from global memory directly each
// load's 64 lanes would touch ~40 cache lines (and a CU's wavefronts together
// more lines than its L1 holds); staged, the rows come in and go out by loads
// and stores of consecutive doubles across the lanes.  The factors and scan
// products stay in registers from row to row (they are five times a row's own
// bytes), and the next row is on its way while one is solved.
__device__ __forceinline__ void tri_rows_staged(int n, int w, const double *__restrict__ Y, double *__restrict__ C,
                                       long long ystride, int r0, int step, int rend, const double *__restrict__ fac,
                                       double *sa, double *sb)
{
    const int lane = threadIdx.x & 63;
    const int keep = fac_keep(n), lo = w * keep, hi = lo + keep < n ? lo + keep : n;
    const TriLane t = tri_lane(n, lo, hi);
    const double *ih = fac + (size_t)fac_windows(n) * kFacStride;
    const int base = t.wa - 1, cnt = t.wb - base + 1;  // y[wa - 1 .. wb]
    double v[kTriPass], g[kRun], ial[kRun], gb;
    if (r0 < rend) load_span(v, Y + r0 * ystride + base, cnt);
    tri_factor_load(fac, w, g, ial, gb);
    for (int k = threadIdx.x; k < cnt - 1; k += blockDim.x) sb[k] = ih[base + k];  // ih[wa - 1 .. wb - 1]
    const TriScan S = tri_scan(g, gb);
    __syncthreads();
    for (int r = r0; r < rend; r += step) {
        store_span(sa, v, cnt);
        wave_lds_sync();
        if (r + step < rend) load_span(v, Y + (r + step) * ystride + base, cnt);
        const OutLds o{sa, lo};  // the staged row is all read before the first kept row is written
        tri_solve<SplineRhsLds, false>(n, SplineRhsLds{sa, sb, base}, lo, hi, o, t, g, ial, gb, S, IhLds{sb, base});
        wave_lds_sync();
        double *out = C + r * ystride + lo;
#pragma unroll
        for (int p = 0; p < kTriPass; p++) {
            const int k = p * 64 + lane;
            if (k < hi - lo) out[k] = sa[k];
        }
        wave_lds_sync();
    }
}

// ---- the fslength table's spline: knots evenly spaced but for their rounding ----
// With one spacing h the factors need no knots: alp_i = h / gam_i, gam_i = 1 /
// (4 - gam_{i-1}) from gam_0 = 0, at its limit 2 - sqrt(3) to the last bit by
// row 16.  The stored knots differ from even ones by their rounding, d <= 4e-16
// in x; what that changes in the factors (relative d / h) reaches the spline's
// values as h^2 c d / h, below what d itself changes in them, dy/dx d.  The
// right-hand side, where a second difference would magnify it, takes each
// interval's own length: 1 / h corrected by one Newton step (relative (d /
// h)^2).  Small solves wait for a chain of divisions in the general factors:
// 1600 knots 11.6 us with them.
// The knots count as even (uniform_even) where (d / h)^2 is below a rounding: h
// at least 2^25 units in the last place of x, 1.4e-7 at log a = -4.6.  Closer
// ones (2000 steps within 0.5% of the starting a) take the general factors and
// divisions: with the constant ones the values of 80 knots over 1e-10 in log a
// were off by 4e-10 of the largest, over 1e-6 by 1e-18.
__device__ __forceinline__ bool uniform_even(const UniformKnots &kn)
{
    return kn.span * kn.rden >= 0x1p-25 * fmax(fabs(kn.x0), fabs(kn.x0 + kn.span));
}
constexpr int kGamRows = 20;
struct GamTab {
    double g[kGamRows + 1];
    constexpr GamTab() : g()
    {
        for (int i = 1; i <= kGamRows; i++) g[i] = 1.0 / (4.0 - g[i - 1]);
    }
};
static_assert(kGamRows == 2 * kRun, "rows 1 .. 20 are those of a first window's lanes 0 and 1");

struct UniformRhsLds {
    const double *ys;
    UniformKnots kn;
    double ih0;
    int base;
    __device__ __forceinline__ double slope(double xl, double xr, double yl, double yr) const
    {
        return (yr - yl) * fma(fma(xl - xr, ih0, 1.0), ih0, ih0);
    }
    __device__ __forceinline__ double operator()(int i) const
    {
        const int k = i - base;
        const double xm = kn.at(i), ym = ys[k];
        return 3.0 * (slope(xm, kn.at(i + 1), ym, ys[k + 1]) - slope(kn.at(i - 1), xm, ys[k - 1], ym));
    }
};
// The same on any knots x, in memory.
struct KnotsRhsLds {
    const double *ys, *x;
    int base;
    __device__ __forceinline__ double slope(int i) const  // of interval i
    {
        const double h = x[i + 1] - x[i];
        return h != 0.0 ? (ys[i + 1 - base] - ys[i - base]) * (1.0 / h) : 0.0;
    }
    __device__ __forceinline__ double operator()(int i) const { return 3.0 * (slope(i) - slope(i - 1)); }
};
struct NoIh {
    __device__ __forceinline__ double operator()(int) const { return 0.0; }
};

// Window w (of fac_windows(n), n >= 3) of the fslength table's coefficients c
// by one wavefront; x: the knots as stored; sa: kTriSpan doubles of its own LDS.
template <bool EVEN>
__device__ __forceinline__ void uniform_spline_form(const UniformKnots &kn, const double *x, const double *__restrict__ y,
                                                    double *__restrict__ c, int n, int w, double *sa)
{
    constexpr GamTab kGam;
    const int lane = threadIdx.x & 63;
    const int keep = fac_keep(n), lo = w * keep, hi = lo + keep < n ? lo + keep : n;
    const TriLane t = tri_lane(n, lo, hi);
    const int base = t.wa - 1, cnt = t.wb - base + 1;  // y[wa - 1 .. wb]
    double v[kTriPass], g[kRun], ial[kRun], before, ih0 = 0.0;
    load_span(v, y + base, cnt);
    if constexpr (EVEN) {
        ih0 = 1.0 / (kn.span * kn.rden);
        // rows 1 .. 20 of a first window (its rows start at 1; the other windows' start beyond 20)
        const bool l0 = t.wa == 1 && lane == 0, l1 = t.wa == 1 && lane == 1;
#pragma unroll
        for (int j = 0; j < kRun; j++) {
            const double gj = l0 ? kGam.g[1 + j] : (l1 ? kGam.g[kRun + 1 + j] : kGam.g[kGamRows]);
            g[j] = j < t.len ? gj : 0.0;
            ial[j] = g[j] * ih0;
        }
        before = lane == 0 ? 0.0 : (l1 ? kGam.g[kRun] : kGam.g[kGamRows]);
    } else {
        tri_factor(x, t, g, ial, before);
    }
    const TriScan S = tri_scan(g, before);
    store_span(sa, v, cnt);
    wave_lds_sync();
    // the staged row is all read before the first kept row is written
    if constexpr (EVEN)
        tri_solve<UniformRhsLds, false>(n, UniformRhsLds{sa, kn, ih0, base}, lo, hi, OutLds{sa, lo}, t, g, ial, before,
                                        S, NoIh{});
    else
        tri_solve<KnotsRhsLds, false>(n, KnotsRhsLds{sa, x, base}, lo, hi, OutLds{sa, lo}, t, g, ial, before, S,
                                      NoIh{});
    wave_lds_sync();
#pragma unroll
    for (int p = 0; p < kTriPass; p++) {
        const int k = p * 64 + lane;
        if (k < hi - lo) c[lo + k] = sa[k];
    }
}

__device__ __forceinline__ void uniform_spline_wave(const UniformKnots &kn, const double *x, const double *__restrict__ y,
                                                    double *__restrict__ c, int n, int w, double *sa)
{
    if (uniform_even(kn)) uniform_spline_form<true>(kn, x, y, c, n, w, sa);
    else uniform_spline_form<false>(kn, x, y, c, n, w, sa);
}

// ---- derivatives for the adjoint ----------------------------------------

// j0'(z) = (z cos z - sin z) / z^2, Taylor series below |z| = 0.5
__device__ __forceinline__ double sph_j0_prime(double z)
{
    if (fabs(z) < 0.5) {
        const double y = z * z;
        // d/dz of 1 - z^2/6 + z^4/120 - z^6/5040 + z^8/362880 - z^10/39916800 + z^12/6227020800
        return z * (-2.0 / 6.0 + y * (4.0 / 120.0 + y * (-6.0 / 5040.0 + y * (8.0 / 362880.0 +
                    y * (-10.0 / 39916800.0 + y * (12.0 / 6227020800.0))))));
    }
    double s, c;
    sincos(z, &s, &c);
    return (z * c - s) / (z * z);
}

// specialJ(x, qc) with its partial derivatives d/dx and d/dqc.
template <bool HYB = true>
__device__ inline double specialJ_d(double x, const JPar &P, double &dJdx, double &dJdqc)
{
    if (HYB && P.qc > 0) {
        const double qc = P.qc;
        const double z = qc * x;
        double s, c;
        sincos(z, &s, &c);
        const double j0 = fabs(z) < 0.5 ? sph_j0(z) : s / z;
        const double j0p = sph_j0_prime(z);
        double J = 0.0, Jx = 0.0, Jq = 0.0;
        for (int n = 1; n < 20; n++) {
            const double nn = (double)(n * n), d = nn + x * x, rd = rcp_fast(d);
            const double A = (n * n + n * n * n * qc + n * qc * x * x - x * x);
            const double B = (2 * n + n * n * qc + qc * x * x);
            const double ii = A * qc * j0 + B * c;
            const double Ax = 2.0 * n * qc * x - 2.0 * x, Bx = 2.0 * qc * x;
            const double Aq = (double)(n * n * n) + n * x * x, Bq = nn + x * x;
            const double iix = Ax * qc * j0 + A * qc * qc * j0p + Bx * c - B * qc * s;
            const double iiq = Aq * qc * j0 + A * (j0 + z * j0p) + Bq * c - B * x * s;
            const double sgn = (n & 1) ? 1.0 : -1.0;
            const double w = sgn * P.en[n] * (rd * rd);
            J += w * ii;
            Jx += w * (iix - 4.0 * x * rd * ii);
            Jq += w * (iiq - n * ii);
        }
        const double Z = 1.5 * 1.202056903159594 * (1 - P.nufrac_low);
        dJdx = Jx / Z;
        dJdqc = Jq / Z;
        return J / Z;
    }
    dJdqc = 0.0;
    if (x <= 0.) {
        dJdx = 0.0;
        return 1.;
    }
    const double x2 = x * x, x3 = x2 * x, x4 = x2 * x2, x7 = x4 * x3, x8 = x4 * x4;
    const double p = pow_fit(x);
    const double N = 1. + 0.0168 * x2 + 0.0407 * x4;
    const double D = 1. + 2.1734 * x2 + 1.6787 * p + 0.1467 * x8;
    const double Nx = 0.0336 * x + 0.1628 * x3;
    // below pow_fit's range p stays finite where x^4.1811 / x goes to nothing
    const double px = x < 0x1p-64 ? 0.0 : p / x;
    const double Dx = 4.3468 * x + 1.6787 * 4.1811 * px + 1.1736 * x7;
    dJdx = (Nx * D - N * Dx) / (D * D);
    return N / D;
}

// Weights of S(x) = y_i + dx (b + dx (c_i + dx d)) on y_i, y_{i+1}, c_i, c_{i+1}.
__device__ __forceinline__ void cspline_grad(double xl, double xr, double x, double &wy0, double &wy1, double &wc0,
                                             double &wc1)
{
    const double h = xr - xl, dx = x - xl, ih = rcp_fast(h);
    const double t = dx * ih, dx3 = dx * dx * dx * ih * (1.0 / 3.0);
    wy0 = 1.0 - t;
    wy1 = t;
    wc0 = -dx * h * (2.0 / 3.0) + dx * dx - dx3;
    wc1 = -dx * h * (1.0 / 3.0) + dx3;
}

}  // namespace kn_dnu

#endif
