// tridiag_device.h -- implicit QL iteration of a symmetric tridiagonal matrix
// by one wave (the iteration of tql2, ED_GREENS_FUNCTIONS.f90:361-499).
//
// The recurrence over the rotations is serial, so all 64 lanes carry the same
// scalars; they share the scan for a negligible off-diagonal element and the
// shift of the diagonal.  d[0..n), e[0..n) (e[i] couples i and i + 1,
// e[n-1] = 0) are in LDS, scaled to entries of at most 1 (ql_scale).
//
// Bound by the latency of a rotation's dependent operations, so its body has
// no branch: a rotation of two numbers below 1e-140 is replaced by the
// identity through selects, and only lane 0's stores go to the arrays (the
// other lanes store to a slot of their own, without masking).
#pragma once

#include <hip/hip_runtime.h>

namespace dmed {

// LDS written by one lane is read by the others of its wave: the hardware
// keeps a wave's LDS operations in order, this keeps the compiler's
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// 1/sqrt(x) for normal x well inside the range.  With e = 1 - x y^2 of the
// hardware estimate y, 1/sqrt(x) = y (1 - e)^(-1/2) = y (1 + e/2 + 3 e^2/8 + ..):
// the terms kept leave e^3, far below rounding, in four dependent operations
// (the recurrence below waits for every one of them).
__device__ __forceinline__ double rsqrt_series(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// first m >= l with a negligible e[m]
__device__ __forceinline__ int ql_find(const double *e, int n, int l, double tst1)
{
    const int lane = threadIdx.x & 63;
    for (int i0 = l; i0 < n; i0 += 64) {
        const bool hit = i0 + lane < n && tst1 + fabs(e[min(i0 + lane, n - 1)]) == tst1;
        const unsigned long long b = __ballot(hit);
        if (b) return i0 + __ffsll(b) - 1;
    }
    return n - 1;
}

// power of two that brings the entries of d[0..n), e[0..n) to at most 1 in
// magnitude, 1 for a zero matrix; exact to multiply and divide by
__device__ __forceinline__ double ql_scale(const double *d, const double *e, int n)
{
    double a = 0.0;
    for (int i = threadIdx.x & 63; i < n; i += 64) a = fmax(a, fmax(fabs(d[i]), fabs(e[i])));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) a = fmax(a, __shfl_xor(a, off, 64));
    return a > 0.0 ? ldexp(1.0, -ilogb(a) - 1) : 1.0;
}

// doubles of `sink` below
constexpr int kQlSink = 64;

// One QL iteration on rows l..m (l < m); f accumulates the shifts.  ROT: the
// rotations, i = m-1 down to l, are stored in rc[i], rs[i]; else they are
// applied to the row z[0..n).  sink: kQlSink doubles of LDS.  Returns |e[l]|
// afterwards.
template <bool ROT>
__device__ __forceinline__ double ql_iterate(double *d, double *e, int n, int l, int m, double &f,
                                             double *rc, double *rs, double *z, double *sink)
{
    const int lane = threadIdx.x & 63;
    const double el = e[l], dl = d[l], el1 = e[l + 1];
    double p = (d[l + 1] - dl) / (2.0 * el);
    // p plus its sign times sqrt(p^2 + 1), without overflow
    double r = fabs(p) < 1e150 ? sqrt(p * p + 1.0) : fabs(p);
    const double pr = p + (p >= 0.0 ? r : -r);
    const double nl = el / pr, dl1 = el * pr, sh = dl - nl;
    wave_lds_fence();
    if (lane == 0) {
        d[l] = nl;
        d[l + 1] = dl1;
    }
    for (int i = l + 2 + lane; i < n; i += 64) d[i] -= sh;
    wave_lds_fence();
    f += sh;
    p = d[m];
    double c = 1.0, c2 = 1.0, c3 = 1.0, s = 0.0, s2 = 0.0;
    double ei = e[m - 1], di = d[m - 1], zn = 0.0, zi = 0.0;
    if constexpr (!ROT) {
        zn = z[m];
        zi = z[m - 1];
    }
    const int step = lane == 0 ? 1 : 0;
    double *pe = lane == 0 ? e + m : sink + lane, *pd = lane == 0 ? d + m : sink + lane;
    double *p1 = lane == 0 ? (ROT ? rc + m - 1 : z + m) : sink + lane;
    double *p2 = lane == 0 && ROT ? rs + m - 1 : sink + lane;
    for (int i = m - 1; i >= l; --i) {
        // the next rotation's operands are loaded ahead of this one's use
        const int in = i > l ? i - 1 : l;
        const double en = e[in], dn = d[in];
        double zp = 0.0;
        if constexpr (!ROT) zp = z[in];
        c3 = c2;
        c2 = c;
        s2 = s;
        const double g = c * ei, h = c * p;
        const double h2 = fma(p, p, ei * ei);
        const bool ok = h2 > 1e-280;
        const double inv = rsqrt_series(ok ? h2 : 1.0);
        r = h2 * inv;
        const double eo = s * r;
        s = ok ? ei * inv : 0.0;
        c = ok ? p * inv : 1.0;
        p = c * di - s * g;
        const double dout = h + s * (c * g + s * di);
        *pe = eo;
        *pd = dout;
        if constexpr (ROT) {
            *p1 = c;
            *p2 = s;
            p2 -= step;
        } else {
            *p1 = s * zi + c * zn;
            zn = c * zi - s * zn;
            zi = zp;
        }
        pe -= step;
        pd -= step;
        p1 -= step;
        ei = en;
        di = dn;
    }
    p = -s * s2 * c3 * el1 * e[l] / dl1;
    const double nel = s * p;
    wave_lds_fence();
    if (lane == 0) {
        e[l] = nel;
        d[l] = c * p;
        if constexpr (!ROT) z[l] = zn;
    }
    wave_lds_fence();
    return fabs(nel);
}

}  // namespace dmed
