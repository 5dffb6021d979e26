// cfdmx_bicg.hpp -- what the launched BiCGSTAB phases (cfdmx_kernels.hip) and the resident
// kernel (cfdmx_bicg_grid.hip) share.
#pragma once
#include "cfdmx_internal.hpp"

namespace cfdmx {

// planes of march block `chunk`: first plane and direction
__device__ __forceinline__ void march_span(const Geo &g, int chunk, int &first, int &dir, int &len)
{
    const int i0 = chunk * kChunk, i1 = min(i0 + kChunk, g.nxc);
    len = i1 - i0;
    dir = (chunk & 1) ? 1 : -1;
    first = dir > 0 ? i0 : i1 - 1;
}

// one row of the operator from the 1-D coefficients of its cell
// What the diagonal leaves out: a coefficient towards a neighbour that does not exist, else
// 0.0 (taking 0.0 off, or adding -0.0 to, a sum of positive terms changes nothing).
struct RowEnds {
    double xm, xp, ym, yp, zm, zp;
};
template <int PRE>
__device__ __forceinline__ double march_diag(const RowEnds &end, double xm, double xp, double ym,
                                             double yp, double zm, double zp)
{
    double ijk = xm + ym + zm + xp + yp + zp;
    if (PRE == 0) {
        ijk -= end.xm;
        ijk -= end.xp;
        ijk -= end.ym;
        ijk -= end.yp;
        ijk -= end.zm;
        ijk -= end.zp;
    } else {
        // one of the two per axis, the upper one where both are missing
        const double aa = end.xp != 0.0 ? -end.xp : -end.xm;
        const double bb = end.yp != 0.0 ? -end.yp : -end.ym;
        const double cc = end.zp != 0.0 ? -end.zp : -end.zm;
        ijk = ijk + aa + bb + cc;
    }
    return ijk;
}
// the six couplings; PRE = 1: scaled by jp, the reciprocal of the diagonal
template <int PRE>
__device__ __forceinline__ void march_offdiag(double xm, double xp, double ym, double yp,
                                              double zm, double zp, double jp, double v[7])
{
    if (PRE == 0) {
        v[0] = -xm;
        v[1] = -yp;
        v[2] = -zm;
        v[4] = -zp;
        v[5] = -ym;
        v[6] = -xp;
    } else {
        v[0] = -xm * jp;
        v[1] = -ym * jp;
        v[2] = -zm * jp;
        v[4] = -zp * jp;
        v[5] = -yp * jp;
        v[6] = -xp * jp;
    }
}
template <int PRE>
__device__ __forceinline__ void march_row(const RowEnds &end, double xm, double xp, double ym,
                                          double yp, double zm, double zp, double v[7])
{
    const double ijk = march_diag<PRE>(end, xm, xp, ym, yp, zm, zp);
    const double jp = PRE ? 1.0 / ijk : 0.0;
    march_offdiag<PRE>(xm, xp, ym, yp, zm, zp, jp, v);
    v[3] = PRE ? ijk * jp : ijk;
}

// The scalars of iteration m > 0 from the end of iteration m-1 (bicgstabRe2.hpp:129-174),
// t = (r,r), (r,r0).  False when the solve has ended.
struct BicgNext {
    double res, beta;
    int mode;
};
__device__ __forceinline__ bool bicg_next(const double (&t)[2], double norm0, double tol,
                                          double restart_factor, int maxit, int timestep, int m,
                                          double alpha, double omega, double rho_l, BicgNext &o)
{
    o.res = sqrt(t[0]) / norm0;                    // L2Norm(r1) / norm0
    if (o.res < tol || m - 1 >= maxit) return false; // m - 1: pIter of the iteration that ended
    o.beta = (alpha / omega) * (t[1] / rho_l);
    o.mode = (timestep < 10 || fabs(rho_l) > tol * restart_factor) ? 0 : 1;
    return true;
}

// v when ok is 1, +0 when ok is 0, by masking the bits (a select here becomes a branch
// around the LDS store, which costs the plane loop its overlap of loads and stores)
__device__ __forceinline__ double keep_if(double v, int ok)
{
    return __longlong_as_double(__double_as_longlong(v) & -(long long)ok);
}
__device__ __forceinline__ float keep_if(float v, int ok)
{
    return __int_as_float(__float_as_int(v) & -ok);
}

} // namespace cfdmx
