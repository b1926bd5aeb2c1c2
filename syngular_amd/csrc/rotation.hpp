// Jacobi rotations of the two-sided Gram eigen-solvers.
#pragma once
#include "common.hpp"

namespace syn {

// Rotation test of plane (p, q): |G_pq| > max(tol sqrt(|G_pp G_qq|), floor),
// in squares (no square root on the critical path of a round), for a matrix
// whose largest diagonal entry is within 1e-100 .. 1e100: beyond, the squares
// leave the range of doubles and the test would find nothing to rotate.
__device__ __forceinline__ bool rotates(double apq, double app, double aqq, double tol, double floor_abs) {
    const double a2 = apq * apq;
    return a2 > tol * tol * fabs(app * aqq) && fabs(apq) > floor_abs;
}

// The same at any scale, for entries in memory that are not scaled beforehand:
// floor is eps max G_ii, so it tells whether a power of two has to bring the
// entries into that range.  The choice is the same for all planes of a matrix.
// The LDS kernels scale their matrix once instead (an order-16 matrix takes 55 us
// so, 59 with this form).
__device__ __forceinline__ bool rotates_any(double apq, double app, double aqq, double tol, double floor_abs) {
    if (floor_abs < 1e-130 || floor_abs > 1e120) {
        const double f = floor_abs < 1.0 ? 0x1p700 : 0x1p-700;
        const double a = f * apq;
        return a * a > tol * tol * fabs(f * app * (f * aqq)) && fabs(apq) > floor_abs;
    }
    return rotates(apq, app, aqq, tol, floor_abs);
}

// Even power of two that brings a matrix of largest diagonal entry m into the
// range of `rotates` (0 where it is in it, or zero, or not finite).
__device__ __forceinline__ int gram_shift(double m) {
    const bool in = m >= 1e-100 && m <= 1e100;
    return in || !(m > 0.0) || m > __DBL_MAX__ ? 0 : -(ilogb(m) & ~1);
}

// Jacobi rotation annihilating G_pq (Rutishauser's angle, Golub & Van Loan
// 8.5.2): with d = G_qq - G_pp and e = 2 G_pq, tau = d / e and
// t = sign(tau) / (|tau| + sqrt(1 + tau^2)) = sign(d e) |e| / (|d| + sqrt(d^2 + e^2)),
// c = 1 / sqrt(1 + t^2), s = c t.  The scaled form needs one division and one
// square root for t; operands far from 1 (|d|, |e| outside 1e-150 .. 1e150)
// take the tau form, which cannot overflow.
// 1 / x and 1 / sqrt(x) for normal positive x from the hardware estimates
// (v_rcp_f64, v_rsq_f64) and two Newton-Raphson steps each: r <- r + r (1 - x r)
// and y <- y + y (1 - x y^2) / 2, each step squaring the relative error, to
// within a unit or two in the last place.  The rotation needs c^2 + s^2 = 1 to
// that level, not correctly rounded c and s; the steps are shorter than the
// IEEE division and square root sequences on a round's critical path.
__device__ __forceinline__ double recip_nr(double x) {
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
}

__device__ __forceinline__ double rsqrt_nr(double x) {
    double y = __builtin_amdgcn_rsq(x);
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const double e = fma(-x * y, y, 1.0);
        y = fma(0.5 * y, e, y);
    }
    return y;
}

__device__ __forceinline__ void rotation(double apq, double app, double aqq, double &c, double &s) {
    const double d = aqq - app, e = 2.0 * apq;
    const double ad = fabs(d), ae = fabs(e), m = fmax(ad, ae);
    double t;
    if (m < 1e150 && m > 1e-150) {
        const double h2 = fma(d, d, e * e);
        t = copysign(ae, d * e) * recip_nr(ad + h2 * rsqrt_nr(h2));
    } else {
        const double tau = d / e, at = fabs(tau);
        t = copysign(1.0, tau) / (at < 1e150 ? at + sqrt(fma(at, at, 1.0)) : 2.0 * at);
    }
    c = rsqrt_nr(fma(t, t, 1.0));
    s = c * t;
}

}  // namespace syn
