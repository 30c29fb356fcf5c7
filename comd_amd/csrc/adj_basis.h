// adj_basis.h -- the Chebyshev basis sums shared by the adjoint kernels
// (csrc/adjoint.hip over link cells, csrc/nlist.hip over the neighbour
// lists).  Series in the convention of src-flat/cheby.c:290-310.
#pragma once

#include "comd_internal.h"

#include <type_traits>

#define AMAX 32   // coefficients per series supported by the adjoint
#define ANMOM 64  // moments written per block (two sets of AMAX)

// The sums below run over NC terms, the series' stride (the coefficients
// padded to a multiple of 8; the caller ignores a[k] past its own count).
// The count is the kernel's own, one instance for each: with a test of k in
// every term each term was a block of its own for the scheduler, and the
// recurrences ran at their latency (16 x 32 000 atoms of 32 terms, mixed:
// the list passes 384, 338, 230 us, now 332, 258, 194 with wave_sums below).

// T_0..T_{NC-1} at y, each times wa added to a[] (and times wb to b[]).
template <int MIXED, int TWO, int NC>
__device__ __forceinline__ void add_basis(double y, double wa, double wb, double *a, double *b)
{
    using T = typename std::conditional<MIXED != 0, float, double>::type;
    const T yt = (T)y, y2 = (T)2 * yt;
    T tm = (T)1, t = yt;
    a[0] += wa;
    if (TWO) b[0] += wb;
#pragma unroll
    for (int k = 1; k < NC; k++) {
        a[k] += wa * (double)t;
        if (TWO) b[k] += wb * (double)t;
        const T tn = y2 * t - tm;
        tm = t;
        t = tn;
    }
}

// add_basis<MIXED, 0, NC> that also returns the series c at y from the same
// basis values: c_0 / 2 + sum_k c_k T_k(y) (the convention of
// src-flat/cheby.c:290-310; c zero-padded to NC, at an address common to
// the wave), in place of a separate Clenshaw sum over the same argument.
template <int MIXED, int NC>
__device__ __forceinline__ double add_basis_sum(double y, double wa, double *a, const double *cg)
{
    using T = typename std::conditional<MIXED != 0, float, double>::type;
    const CM_CONST double *c = (const CM_CONST double *)cg;
    double s = 0.5 * c[0];
    const T yt = (T)y, y2 = (T)2 * yt;
    T tm = (T)1, t = yt;
    a[0] += wa;
#pragma unroll
    for (int k = 1; k < NC; k++) {
        a[k] += wa * (double)t;
        s += c[k] * (double)t;
        const T tn = y2 * t - tm;
        tm = t;
        t = tn;
    }
    return s;
}

// T_k(y) times wt plus the derivative of T_k with respect to y, k U_{k-1}(y)
// (U: the second-kind polynomials, U_0 = 1, U_1 = 2y), times wd, added to
// a[k], k < NC.  With wd = w / (b - a) (the domain's dy/dr = 2 / (b - a)
// times w / 2) this is, for the series' basis B_k (B_0 = T_0 / 2 applied by
// the caller), the pair's term of the energy moments and of the derivative
// operator applied to the force moments in one set.  In FP64 the derivatives
// have their own recurrence, T'_{k+1} = 2 T_k + 2y T'_k - T'_{k-1}: the same
// operations per term, without the constants k held in registers.
template <int MIXED, int NC>
__device__ __forceinline__ void add_basis_deriv(double y, double wt, double wd, double *a)
{
    a[0] += wt;
    if constexpr (MIXED) {
        const float yf = (float)y, y2 = 2.0f * yf;
        float tm = 1.0f, t = yf, um = 1.0f, u = y2;  // T_{k-1}, T_k, U_{k-1}, U_k at k = 1
#pragma unroll
        for (int k = 1; k < NC; k++) {
            a[k] += wt * (double)t;
            a[k] += wd * (double)k * (double)um;
            const float tn = y2 * t - tm, un = y2 * u - um;
            tm = t;
            t = tn;
            um = u;
            u = un;
        }
    } else {
        const double y2 = 2.0 * y;
        double tm = 1.0, t = y, vm = 0.0, v = 1.0;  // T_{k-1}, T_k and their derivatives at k = 1
#pragma unroll
        for (int k = 1; k < NC; k++) {
            a[k] += wt * t;
            a[k] += wd * v;
            const double vn = 2.0 * t + (y2 * v - vm), tn = y2 * t - tm;
            vm = v;
            v = vn;
            tm = t;
            t = tn;
        }
    }
}

__device__ __forceinline__ double cheb_arg(double x, double a, double b)
{
    if (x < a) x = a;  // lower clamp only (src-flat/cheby.c:290-293)
    return (2.0 * x - a - b) / (b - a);
}

// Sum of v over the wave's 64 lanes (result in every lane).
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Sums of a[0 .. 32) over the wave's 64 lanes: lanes 2k and 2k + 1 get that of
// a[k].  At each step a lane keeps half of its values and gives the others to
// the lane it is paired with, 32 exchanges in all where a sum per value
// takes 192 and 160 more additions.  a is overwritten.
__device__ __forceinline__ double wave_sums(double (&a)[AMAX])
{
    const int L = threadIdx.x & 63;
#pragma unroll
    for (int h = AMAX / 2; h > 0; h >>= 1) {
        // lane bit 2h selects the half that the lane keeps
        const bool up = (L & (2 * h)) != 0;
#pragma unroll
        for (int k = 0; k < h; k++) {
            const double lo = a[k], hi = a[k + h];
            a[k] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, 2 * h, 64);
        }
    }
    return a[0] + __shfl_xor(a[0], 1, 64);
}

// The moments a[k] summed over the block's waves, in wave order through LDS
// (red: one row of ANMOM doubles per wave), and written by threads 0 .. 63
// to part[0 .. ANMOM): a block's partials in a fixed order.  SET 0: a[] is
// the first set of AMAX moments, the second is zero; SET 1: the reverse.
template <int SET>
__device__ __forceinline__ void block_moments(double (&a)[AMAX], double (*red)[ANMOM], double *part)
{
    const int L = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const double s = wave_sums(a);
    red[w][(L & 1 ? 1 - SET : SET) * AMAX + (L >> 1)] = L & 1 ? 0.0 : s;
    __syncthreads();
    if (threadIdx.x < ANMOM) {
        double s = 0.0;
        for (int q = 0; q < nw; q++) s += red[q][threadIdx.x];
        part[threadIdx.x] = s;
    }
}
