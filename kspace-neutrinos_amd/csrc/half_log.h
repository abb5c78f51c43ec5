// half_log.h -- log(sqrt(k2)) of an integer, for the rescale sweep.
#ifndef KN_HALF_LOG_H
#define KN_HALF_LOG_H

#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>

#include "kn_logtab.h"

namespace kn_res {

// log(sqrt(k2)), k2 >= 1, by kn_logtab: k2 = 2^e m with m in the table's
// interval j, log m = -log r_j + log1p(m r_j - 1) with six terms of the series
// (|m r_j - 1| <= 2^-8: the seventh is below 2e-18).  e log(2) / 2 to 44 digits
// plus the table's entry is exact, and what is added to it is below 2e-3, so
// the sum's rounding is all but the whole error: half a unit in the last place
// plus 1e-17, at most 0.90e-15 over all int k2.  (0.89e-15 for half of a
// correctly rounded log(k2); with entries and sums rounded on the way, 1.76e-15.)
// 17 operations where the math library's log and its double-double steps are
// about 75.
__device__ __forceinline__ double half_log(int k2, const double2 *lg)
{
    const double d = (double)k2;
    long long v;
    __builtin_memcpy(&v, &d, sizeof v);
    const int hi = (int)(v >> 32), e = (hi >> 20) - 1023;
    const long long mv = (v & 0x000fffffffffffffLL) | 0x3ff0000000000000LL;
    double m;
    __builtin_memcpy(&m, &mv, sizeof m);
    const double2 t = lg[(hi >> 13) & (KN_LOGTAB_N - 1)];
    const double r = fma(m, t.x, -1.0), ef = (double)e;
    double q = fma(r, -1.0 / 6.0, 1.0 / 5.0);
    q = fma(r, q, -1.0 / 4.0);
    q = fma(r, q, 1.0 / 3.0);
    q = fma(r, q, -1.0 / 2.0);
    const double p = fma(r * r, q, r);
    return fma(ef, KN_HALF_LN2_HI, t.y) + fma(ef, KN_HALF_LN2_LO, 0.5 * p);
}

}  // namespace kn_res

#endif
