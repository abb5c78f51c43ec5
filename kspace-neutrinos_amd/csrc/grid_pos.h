// grid_pos.h -- places of modes on a rank's slabs, shared by the grid sweeps.
#ifndef KN_GRID_POS_H
#define KN_GRID_POS_H

#include <hip/hip_runtime.h>

namespace kn_grid {

// KVAL of powerspectrum.c:27
__host__ __device__ inline int kval(int n, int dims) { return n <= dims / 2 ? n : n - dims; }

struct Pos {
    int i, j, z;  // slab, row and z of a mode
};

// Position of mode m of the rank's slabs.
__device__ __forceinline__ Pos pos_of(long long m, int rowlen, int dims)
{
    Pos p;
    if (m < 0x7fffffffLL) {  // 32-bit divisions
        const unsigned r = (unsigned)m / (unsigned)rowlen;
        p.z = (int)((unsigned)m - r * (unsigned)rowlen);
        p.j = (int)(r % (unsigned)dims);
        p.i = (int)(r / (unsigned)dims);
    } else {
        const long long r = m / rowlen;
        p.z = (int)(m - r * rowlen);
        p.j = (int)(r % dims);
        p.i = (int)(r / dims);
    }
    return p;
}

// A step of n modes along the flattened [slab][row][z] order, split so that
// advancing a position costs two compares whatever n is.
struct Step {
    int di, dj, dz;
};

inline Step step_of(long long n, int rowlen, int dims)
{
    const long long r = n / rowlen;
    Step s;
    s.dz = (int)(n % rowlen);
    s.dj = (int)(r % dims);
    s.di = (int)(r / dims);
    return s;
}

__device__ __forceinline__ void advance(Pos &p, const Step &s, int rowlen, int dims)
{
    p.z += s.dz;
    p.j += s.dj;
    p.i += s.di;
    if (p.z >= rowlen) {
        p.z -= rowlen;
        p.j++;
    }
    if (p.j >= dims) {
        p.j -= dims;
        p.i++;
    }
}

}  // namespace kn_grid

#endif
