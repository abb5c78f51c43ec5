// bin_kernels.h -- device kernels of the k-shell binning sweep (a).
//
// Included by powerspectrum.hip.  The kernels are templates over the launch
// shape so the shape can be tuned without touching the arithmetic; the
// arithmetic itself follows powerspectrum.c:56-89 (see powerspectrum.hip).
#ifndef KN_BIN_KERNELS_H
#define KN_BIN_KERNELS_H

#include <hip/hip_runtime.h>
#include <math.h>
#include <vector>

#include "grid_pos.h"
#include "kn_mem.h"

namespace kn_bin {

using kn_grid::Pos;
using kn_grid::Step;
using kn_grid::advance;
using kn_grid::kval;
using kn_grid::pos_of;
using kn_grid::step_of;

// Per-bin smallest |k|^2 reaching the bin under the reference expression
// floor(binsperunit * log(sqrt(k2))) (powerspectrum.c:40, :67).  Returns 0,
// or the first k2 where the expression is not monotone / exceeds nrbins-1.
// thr holds nrbins + 1 ints.
inline long long build_thresholds(int dims, int nrbins, int *thr)
{
    const double binsperunit = (nrbins - 1) / log(sqrt(3) * dims / 2.0);
    const long long kmax2 = 3LL * (dims / 2) * (dims / 2);
    for (int b = 0; b <= nrbins; b++) thr[b] = 0x7fffffff;
    thr[0] = 0;
    int prev = 0;
    for (long long k2 = 1; k2 <= kmax2; k2++) {
        const int b = (int)floor(binsperunit * log(sqrt((double)k2)));
        if (b < prev || b >= nrbins) return k2;
        while (prev < b) thr[++prev] = (int)k2;
    }
    return 0;
}

inline long long build_thresholds(int dims, int nrbins, std::vector<int> &thr)
{
    thr.resize(nrbins + 1);
    return build_thresholds(dims, nrbins, thr.data());
}

// Per-axis inverse CiC window by storage index (powerspectrum.c:8-12); iw holds dims doubles.
inline void build_invwindow(int dims, double *iw)
{
    for (int n = 0; n < dims; n++) {
        const int kx = kval(n, dims);
        iw[n] = kx ? M_PI * kx / (dims * sin(M_PI * kx / (double)dims)) : 1.0;
    }
}

inline void build_invwindow(int dims, std::vector<double> &iw)
{
    iw.resize(dims);
    build_invwindow(dims, iw.data());
}

__device__ __forceinline__ int find_bin(int k2, float half_bpu, const int *__restrict__ thr, int nrbins)
{
    int b = (int)(__logf((float)k2) * half_bpu);
    b = b < 0 ? 0 : (b > nrbins - 1 ? nrbins - 1 : b);
    while (b > 0 && k2 < thr[b]) b--;
    while (b < nrbins - 1 && k2 >= thr[b + 1]) b++;
    return b;
}

__device__ __forceinline__ void advance(Pos &p, int step, int rowlen, int dims)
{
    p.z += step;
    while (p.z >= rowlen) {
        p.z -= rowlen;
        if (++p.j == dims) {
            p.j = 0;
            p.i++;
        }
    }
}

// multiplicity * |F|^2 * ((iwx iwy iwz)^2)^2 in the reference's rounding order
__device__ __forceinline__ double mode_weight(double2 f, double iwxy, double iwz, int kz, int half)
{
    const double w = __dmul_rn(iwxy, iwz);
    const double w2 = __dmul_rn(w, w);
    const double w4 = __dmul_rn(w2, w2);
    const double p2 = __dadd_rn(__dmul_rn(f.x, f.x), __dmul_rn(f.y, f.y));
    double v = __dmul_rn(p2, w4);
    if (kz != 0 && kz != half) v *= 2.0;
    return v;
}

struct BinArgs {
    const double2 *F;
    int dims, startslab, nrbins;
    long long modes;        // of the rank's slabs
    Step in_tile, to_next;  // from a lane's mode to its next one in the block's tile, and from its last one to the next tile's first
    const int *thr;
    const double *iw;
    float half_bpu;
    double *partial;  // gridDim.x * nrbins
    int cshift;       // copies of the bin sums: 2^cshift
};

// Where the sweep keeps its tables: the bin thresholds, the per-axis inverse
// window and the bin sums all in LDS (the fast form); the window read from
// global memory (through the caches) when LDS cannot hold it next to the
// others; or everything in global memory, the bin sums then added with
// global atomics into the block's own partial row (any number of bins).
enum TablePlace { kTablesLds = 0, kWindowGlobal = 1, kTablesGlobal = 2 };

constexpr int kSweepWaves = 8;      // wavefronts per block
constexpr int kSweepUnroll = 2;     // modes per lane of a tile

// LDS bytes of the sweep with `sets` sets of bin sums.
__host__ __device__ constexpr size_t sweep_smem_bytes(int place, int dims, int nrbins, int sets)
{
    return place == kTablesGlobal ? 0
                                  : sizeof(double) * (size_t)nrbins * sets +
                                        sizeof(int) * (size_t)(nrbins + 1 + ((nrbins + 1) & 1)) +
                                        (place == kTablesLds ? sizeof(double) * (size_t)dims : 0);
}

// The bin sweep (powerspectrum.c:56-89).  The grid is cut into tiles of 64
// WAVES U consecutive modes, block b taking tiles b, b + gridDim.x, ...; loads
// are 16 bytes per lane, consecutive across a wavefront, non-temporal (each
// mode is read once per sweep).  A wavefront's place is scalar (WIDE: its 64
// modes lie in at most two rows).  A mode's bin is an fp32 estimate,
// within one of the right one, corrected by the integer thresholds of two
// bins; its weighted power is added to the bin's sum in LDS.  Neighbouring
// lanes often share a bin, and lanes that add to one address wait for each
// other: 2^cshift copies of the sums, taken in turn by the lanes, part them.
// With OWN every wavefront has its own copies and the result is the same on
// every run; without it the block's wavefronts share them, so the order of
// the adds between wavefronts (and the last bit of a sum) can differ from run
// to run.  The block adds the copies in a fixed order into its partial row,
// and k_reduce_partials adds the rows in a fixed order.
// A read at the most this card reaches takes 1.23 ms at 1024^3.  An earlier
// form loaded runs of consecutive modes per lane (a transpose through LDS) to
// merge equal bins before the adds: about 110 vector operations per mode
// where this one has 52, and they, not memory, set its time (1.41 ms at 1024^3
// with the reduction against 1.32).  At 1024^3 one, two and four copies take
// 1548, 1315 and 1320 us; two, three and four blocks per CU 1391, 1315 and 1527.
template <int PLACE, int WAVES, int U, bool OWN, bool WIDE>
__global__ __launch_bounds__(64 * WAVES) void k_bin_sweep(BinArgs a)
{
    constexpr int B = 64 * WAVES, T = B * U;
    const int cshift = PLACE == kTablesGlobal ? 0 : a.cshift, cbyte = cshift + 3;
    extern __shared__ double smem[];
    const int rowlen = a.dims / 2 + 1, half = a.dims / 2, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    long long m = (long long)blockIdx.x * T + 64 * wave;  // the wavefront's first mode
    const long long n = a.modes, S = (long long)gridDim.x * T;
    double2 cur[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const long long mu = m + B * u + lane;
        cur[u] = mu < n ? kn_mem::ld<true>(a.F + mu) : make_double2(0.0, 0.0);
    }
    double *hist = smem;
    const double *iw = a.iw;
    const int *thr = a.thr;
    if constexpr (PLACE == kTablesGlobal) {
        hist = a.partial + (size_t)blockIdx.x * a.nrbins;
        for (int t = threadIdx.x; t < a.nrbins; t += B) hist[t] = 0.0;
    } else {
        const int nhist = ((OWN ? WAVES : 1) * a.nrbins) << cshift;
        int *thr_l = (int *)(hist + nhist);
        for (int t = threadIdx.x; t < nhist; t += B) hist[t] = 0.0;
        for (int t = threadIdx.x; t <= a.nrbins; t += B) thr_l[t] = a.thr[t];
        thr = thr_l;
        if constexpr (PLACE == kTablesLds) {
            double *iw_l = (double *)(thr_l + a.nrbins + 1 + ((a.nrbins + 1) & 1));  // 8-byte aligned
            for (int t = threadIdx.x; t < a.dims; t += B) iw_l[t] = a.iw[t];
            iw = iw_l;
        }
    }
    __syncthreads();
    double *const mine = hist + (OWN ? (wave * a.nrbins) << cshift : 0) + (lane & ((1 << cshift) - 1));
    Pos p = pos_of(m, rowlen, a.dims);
    for (; m < n; m += S) {
        // the wavefront's rows: z of its first mode, kx^2 + ky^2, x and y there and in the next row
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
            int z, k2, x, y;
            if constexpr (WIDE) {
                z = z0[u] + lane;
                const bool next = z >= rowlen;
                z -= next ? rowlen : 0;
                k2 = (next ? kxy[u][1] : kxy[u][0]) + __mul24(z, z);
                x = next ? gx[u][1] : gx[u][0];
                y = next ? gy[u][1] : gy[u][0];
            } else {
                const Pos q = pos_of(mu < n ? mu : 0, rowlen, a.dims);
                x = a.startslab + q.i;
                y = q.j;
                z = q.z;
                const int kx = kval(x, a.dims), ky = kval(y, a.dims);
                k2 = kx * kx + ky * ky + z * z;
            }
            if (mu >= n || k2 == 0) continue;
            int b;
            if constexpr (PLACE == kTablesGlobal) {  // so many bins that the estimate may be further off
                b = find_bin(k2, a.half_bpu, thr, a.nrbins);
            } else {
                b = (int)(__logf((float)k2) * a.half_bpu);
                b = b > a.nrbins - 1 ? a.nrbins - 1 : b;
                const int t0 = thr[b], t1 = thr[b + 1];
                b += (k2 >= t1) - (k2 < t0);
            }
            const double v = mode_weight(cur[u], __dmul_rn(iw[x], iw[y]), iw[z], z, half);
            atomicAdd((double *)((char *)mine + ((unsigned)b << cbyte)), v);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const long long mu = m + S + B * u + lane;
            cur[u] = mu < n ? kn_mem::ld<true>(a.F + mu) : make_double2(0.0, 0.0);
        }
    }
    if constexpr (PLACE != kTablesGlobal) {
        __syncthreads();
        for (int t = threadIdx.x; t < a.nrbins; t += B) {
            double v = 0.0;
            for (int w = 0; w < (OWN ? WAVES : 1); w++)
                for (int c = 0; c < 1 << cshift; c++) v += hist[((w * a.nrbins + t) << cshift) + c];
            a.partial[(size_t)blockIdx.x * a.nrbins + t] = v;
        }
    }
}

}  // namespace kn_bin

#endif
