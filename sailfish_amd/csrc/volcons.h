// volcons.h -- the open-boundary points of obc_volcons (volcons.hip) and their terms.
#pragma once
#include "sf_internal.h"

namespace sf {

template <typename T>
struct VolArgs {
    const T *z, *h, *pm, *pn;
    T *u, *v;
    int szI, szJ;
    int nw, ne, ns, nn;   // points per segment (0 when closed)
};

template <typename T>
__host__ __device__ inline VolArgs<T> vol_args(const T *z, const T *h, const T *pm, const T *pn, T *u, T *v, int szI,
                                               int szJ, int flags)
{
    return VolArgs<T>{z, h, pm, pn, u, v, szI, szJ,
                      (flags & SF_OBC_WEST) ? szJ - 2 : 0, (flags & SF_OBC_EAST) ? szJ - 2 : 0,
                      (flags & SF_OBC_SOUTH) ? szI - 2 : 0, (flags & SF_OBC_NORTH) ? szI - 2 : 0};
}

// segment (0 west, 1 east, 2 south, 3 north) of boundary point b; b becomes its place in it
template <typename T>
__device__ __forceinline__ int vol_segment(const VolArgs<T> &a, int &b)
{
    if (b < a.nw) return 0;
    b -= a.nw;
    if (b < a.ne) return 1;
    b -= a.ne;
    if (b < a.ns) return 2;
    b -= a.ns;
    return 3;
}

// flat index of the velocity point: west / east u points, rows j = 1 .. M-1; south / north
// v points, columns i = 1 .. L-1
template <typename T>
__device__ __forceinline__ long long vol_face(const VolArgs<T> &a, int e, int b)
{
    const long long W = a.szI;
    if (e < 2) return (1 + b) * W + (e == 0 ? 1 : W - 1);
    return (e == 2 ? 1 : a.szJ - 1) * W + 1 + b;
}

// Area term and inflow-signed flux of a face with velocity x between the rho points lo and
// hi (surface z, depth h, metric m along the face); inward: a west or south face.
template <typename T>
__device__ __forceinline__ void vol_terms(T zl, T hl, T zh, T hh, T ml, T mh, T x, bool inward, double &cff, double &fl)
{
    const double len = 2.0 / ((double)ml + (double)mh);
    cff = (0.5 * (((double)zl + (double)hl) + ((double)zh + (double)hh))) * len;
    fl = inward ? cff * (double)x : -(cff * (double)x);
}

}  // namespace sf
