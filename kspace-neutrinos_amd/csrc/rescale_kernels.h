// rescale_kernels.h -- device kernels of the per-mode rescale sweep (c).
//
// Included by rescale.hip.  Arithmetic follows interface_gadget.c:163-188 and
// delta_pow.c:19-37 (see rescale.hip); the templates only vary the launch
// shape and the lane-to-mode mapping.
#ifndef KN_RESCALE_KERNELS_H
#define KN_RESCALE_KERNELS_H

#include <hip/hip_runtime.h>
#include <math.h>
#include <type_traits>

#include "grid_pos.h"
#include "half_log.h"
#include "kn_mem.h"

namespace kn_res {

using kn_grid::Pos;
using kn_grid::Step;
using kn_grid::advance;
using kn_grid::kval;
using kn_grid::pos_of;
using kn_grid::step_of;

struct ResArgs {
    double2 *F;
    int dims, startslab, nbins, nbuckets;
    long long rows;
    long long modes;           // of all rows
    Step in_tile, to_next;     // from a lane's mode to its next one in the block's tile, and from its last one to the next tile's first
    double log_kunit, norm;    // log(2 pi / BoxSize); the ratio's factor
    const double *logkk, *ratio;
    int *nan_flag;
    // Green's function of the PM potential (GREEN sweeps): per axis index t,
    // gw[t] = exp(-kt^2 asmth2) W(t)^-4 (dims doubles; kt the integer
    // wavenumber, W the CiC window, asmth2 = (2 pi r_s / BoxSize)^2)
    const double *__restrict__ gw;
};

// The ints of load_tab: buckets 0 .. nbuckets, in whole doubles.
__host__ __device__ inline int tab_ints(int nbuckets) { return nbuckets + 1 + ((nbuckets + 1) & 1); }

// LDS of the sweep: the logarithm's table (log_lds), the ratio table's log k,
// ratio and slope, its ints, and the Green's factors of one axis.
__host__ __device__ inline size_t smem_bytes(int nbins, int nbuckets, int green_dims, bool log_lds)
{
    return sizeof(double) * (3 * (size_t)nbins + (log_lds ? 2 * KN_LOGTAB_N : 0) + (size_t)green_dims) +
           (nbins > 0 ? sizeof(int) * (size_t)tab_ints(nbuckets) : 0);
}

struct Tab {
    const double *lk, *rt, *sl;  // log k, ratio, and slope of the segment above each bin
    const double2 *lg;           // kn_logtab
    const int *bucket;
    int nbins, nbuckets;
    double x0, x1, inv_bw, norm, log_kunit;
};

// Ratio table, slopes, bucket index and (LOG_LDS) logarithm table into LDS (all threads of the block).
template <bool LOG_LDS>
__device__ __forceinline__ Tab load_tab(const ResArgs &a, int nthreads)
{
    extern __shared__ double sm[];
    double *lk = sm + (LOG_LDS ? 2 * KN_LOGTAB_N : 0), *rt = lk + a.nbins, *sl = rt + a.nbins;
    int *bucket = (int *)(sl + a.nbins);
    if (LOG_LDS)
        for (int t = threadIdx.x; t < 2 * KN_LOGTAB_N; t += nthreads) sm[t] = kn_logtab[t];
    for (int t = threadIdx.x; t < a.nbins; t += nthreads) {
        lk[t] = a.logkk[t];
        rt[t] = a.ratio[t];
    }
    __syncthreads();
    Tab T;
    T.lk = lk;
    T.rt = rt;
    T.sl = sl;
    T.lg = (const double2 *)(LOG_LDS ? sm : kn_logtab);
    T.bucket = bucket;
    T.nbins = a.nbins;
    T.nbuckets = a.nbuckets;
    T.x0 = lk[0];
    T.x1 = lk[a.nbins - 1];
    T.inv_bw = a.nbins > 1 ? a.nbuckets / (T.x1 - T.x0) : 0.0;
    T.norm = a.norm;
    T.log_kunit = a.log_kunit;
    for (int t = threadIdx.x; t < a.nbins; t += nthreads) {
        const double h = t + 1 < a.nbins ? lk[t + 1] - lk[t] : 0.0;
        sl[t] = h > 0.0 ? (rt[t + 1] - rt[t]) / h : 0.0;
    }
    // bucket[q]: the GSL segment index (largest i <= n-2 with lk[i] <= x) at the bucket's left edge
    for (int q = threadIdx.x; q <= a.nbuckets; q += nthreads) {
        const double edge = T.x0 + q / T.inv_bw;
        int lo = 0, hi = a.nbins - 1;
        while (hi > lo + 1) {
            const int mid = (lo + hi) >> 1;
            if (lk[mid] > edge) hi = mid;
            else lo = mid;
        }
        bucket[q] = lo;
    }
    __syncthreads();
    return T;
}

// 1 + get_dnudcdm_powerspec(log(|k|)) for k2 > 0, with |k| = sqrt(k2) 2 pi / BoxSize.
// log|k| is evaluated as log(sqrt(k2)) + log(2 pi / BoxSize): the same value as
// the reference's log(sqrt(k2)*2*M_PI/BoxSize) to about one ulp, without the
// sqrt and the divisions.
// Where the stored slopes do not carry a table (a log k that is not finite, also
// the only bin's; ratios that differ by more than the largest double times the
// bin's width) the result is infinite or NaN; REF is the reference's own
// expression, which needs no slope and may be finite there.
template <bool REF>
__device__ __forceinline__ double smth_of(int k2i, const Tab &T)
{
    double kk = half_log(k2i, T.lg) + T.log_kunit;
    kk = kk < T.x0 ? T.x0 : kk;
    kk = kk > T.x1 ? T.x1 : kk;
    int q = (int)((kk - T.x0) * T.inv_bw);
    q = q < 0 ? 0 : (q > T.nbuckets ? T.nbuckets : q);
    int i = T.bucket[q];
    while (i < T.nbins - 2 && T.lk[i + 1] <= kk) i++;
    if (REF) {
        const double h = T.nbins > 1 ? T.lk[i + 1] - T.lk[i] : 0.0;
        return fma(T.norm, h > 0.0 ? T.rt[i] + (kk - T.lk[i]) / h * (T.rt[i + 1] - T.rt[i]) : T.rt[i], 1.0);
    }
    return fma(T.norm, fma(kk - T.lk[i], T.sl[i], T.rt[i]), 1.0);
}

// The PM Green's function with CiC deconvolution at k2 > 0, as the potential
// pass of a PM step applies it after the neutrino rescale (Gadget-2's
// pmforce_periodic, where the hook of 0002-Add-hooks-to-kspace-neutrino-code.patch:116-125
// calls add_nu_power_to_rhogrid): -exp(-k2 asmth2) / k2 times ff^4, ff the
// product of the three per-axis inverse windows.  exp(-k2 asmth2) factors
// over the axes, so with gw (ResArgs) it is -gw[x] gw[y] gw[z] / k2: no
// exponential per mode, and 1/k2 from the hardware reciprocal refined by one
// Newton step (a few units in the last place from the direct form).
__device__ __forceinline__ double green_of(int k2, double gxy, double gz)
{
    const double d = (double)k2;
    const double r = __builtin_amdgcn_rcp(d);
    const double inv = fma(r, fma(-d, r, 1.0), r);
    return -(gxy * gz) * inv;
}

// The rescale sweep.  The grid is cut into tiles of 64 WAVES U consecutive
// modes, block b taking tiles b, b + gridDim.x, ...: the blocks move over the
// grid together, two of 8 wavefronts per CU, each lane U = 2 modes of a tile
// (loads and stores 16 bytes per lane, consecutive across a wavefront, with the
// non-temporal hint).  HBM bounds it: reading and writing reach the most this
// way (an empty in-place sweep of 1024^3: 5.1-5.5 TB/s from contiguous ranges
// per block, 5.5-6.0 from tiles in turn by 16 wavefronts per CU), but only with
// few operations per mode.  So a wavefront's place is scalar (its 64 modes lie
// in at most two rows, WIDE), log k comes from a table (half_log) and the
// ratio's segment has its slope stored: 77 vector operations per mode against
// 174, a third of the sweep's time.  ms per sweep, contiguous ranges with the
// library's log against this form (Green's function in parentheses): 256^3
// 0.062 -> 0.049 (0.063 -> 0.050), 512^3 0.436 -> 0.360 (0.452 -> 0.365), 768^3
// 1.472 -> 1.250, 1024^3 3.330 -> 3.063 (3.451 -> 3.088), 5.62 TB/s.  At 1024^3
// one, two, three and four blocks per CU take 3.38, 3.07, 3.18 and 3.60 ms, U =
// 1, 3, 4 and 8 3.11, 3.39, 3.38 and 3.41.
// GREEN: the same sweep also applies the Green's function (F s_nu, then times
// G, the two roundings of the two passes it replaces) and zeroes the k = 0
// mode; with nbins 0 it applies the Green's function alone.
// WIDE: rows of 64 modes or more (else every lane finds its own row).
// LOG_LDS: the logarithm's table in LDS (else read through the caches).
template <int WAVES, int U, bool GREEN, bool WIDE, bool LOG_LDS>
__global__ __launch_bounds__(64 * WAVES) void k_rescale(ResArgs a)
{
    constexpr int B = 64 * WAVES, T = B * U;
    const int rowlen = a.dims / 2 + 1, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long m0 = (long long)blockIdx.x * T + 64 * wave;  // the wavefront's first mode
    const long long n = a.modes, S = (long long)gridDim.x * T;
    double2 cur[U];
    auto load = [&](long long m) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const long long mu = m + B * u + lane;
            cur[u] = mu < n ? kn_mem::ld<true>(a.F + mu) : make_double2(0.0, 0.0);
        }
    };
    load(m0);
    Tab Tb;
    const double *gw = nullptr;
    if (!GREEN || a.nbins > 0) Tb = load_tab<LOG_LDS>(a, B);
    if constexpr (GREEN) {
        extern __shared__ double sm[];
        double *gw_l = a.nbins > 0 ? (double *)((int *)(Tb.sl + a.nbins) + tab_ints(a.nbuckets)) : sm;
        for (int t = threadIdx.x; t < a.dims; t += B) gw_l[t] = a.gw[t];
        __syncthreads();
        gw = gw_l;
    }
    bool left = false, saw_nan = false;
    auto sweep = [&](auto ref) {
        Pos p = pos_of(m0, rowlen, a.dims);
        for (long long m = m0; m < n; m += S) {
            // the wavefront's rows: z of its first mode, kx^2 + ky^2 there and in the next row (GREEN: both rows' x and y)
            int z0[U], kxy[U][2], gx[U][2], gy[U][2];
            if constexpr (WIDE) {
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int x0 = a.startslab + p.i;
                    int x1 = x0, j1 = p.j + 1;
                    if (j1 == a.dims) {
                        j1 = 0;
                        x1 = x0 + 1;
                    }
                    const int kx0 = kval(x0, a.dims), ky0 = kval(p.j, a.dims), kx1 = kval(x1, a.dims), ky1 = kval(j1, a.dims);
                    z0[u] = p.z;
                    kxy[u][0] = kx0 * kx0 + ky0 * ky0;
                    kxy[u][1] = kx1 * kx1 + ky1 * ky1;
                    gx[u][0] = x0, gx[u][1] = x1, gy[u][0] = p.j, gy[u][1] = j1;
                    advance(p, u + 1 < U ? a.in_tile : a.to_next, rowlen, a.dims);
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const long long mu = m + B * u + lane;
                int z, k2;
                int x = 0, y = 0;
                if constexpr (WIDE) {
                    z = z0[u] + lane;
                    const bool next = z >= rowlen;
                    z -= next ? rowlen : 0;
                    k2 = (next ? kxy[u][1] : kxy[u][0]) + __mul24(z, z);
                    if constexpr (GREEN) {
                        x = next ? gx[u][1] : gx[u][0];
                        y = next ? gy[u][1] : gy[u][0];
                    }
                } else {
                    const Pos q = pos_of(mu < n ? mu : 0, rowlen, a.dims);
                    const int kx = kval(a.startslab + q.i, a.dims), ky = kval(q.j, a.dims);
                    z = q.z;
                    k2 = kx * kx + ky * ky + z * z;
                    x = a.startslab + q.i;
                    y = q.j;
                }
                if (mu >= n) continue;
                double2 f = cur[u];
                if (k2 <= 0) {
                    if (GREEN) kn_mem::st<true>(a.F + mu, make_double2(0.0, 0.0));
                    continue;
                }
                if (!GREEN || a.nbins > 0) {
                    double s = smth_of<false>(k2, Tb);
                    if (isfinite(s) == decltype(ref)::value) {
                        left = true;
                        continue;
                    }
                    if constexpr (decltype(ref)::value) {
                        s = smth_of<true>(k2, Tb);
                        saw_nan |= isnan(s);
                    }
                    f.x *= s;
                    f.y *= s;
                }
                if constexpr (GREEN) {
                    const double g = green_of(k2, gw[x] * gw[y], gw[z]);
                    f.x *= g;
                    f.y *= g;
                }
                kn_mem::st<true>(a.F + mu, f);
            }
            load(m + S);
        }
    };
    sweep(std::false_type{});
    // the modes that the slopes gave no finite factor, left as they were: a second pass, which all but no table needs (a
    // mark of such tables asked for each mode took 0.3 us of a 128^3 sweep's 9.4, the factor formed again in place 0.1)
    if (__ballot(left)) {
        load(m0);
        sweep(std::true_type{});
    }
    if (saw_nan) atomicOr(a.nan_flag, 1);
}

}  // namespace kn_res

#endif
