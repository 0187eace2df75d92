// Shared by the spline folds on the matrix cores: the 16x16x4 products and the
// sign class of a cubic piece.
#pragma once
#include "xh_common.hpp"

namespace xh {

template <typename R> struct Mfma;

// lane l: A[l % 16][l / 16], B[l / 16][l % 16]; result element r of lane l is
// D[4 r + l / 16][l % 16]
template <> struct Mfma<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4 step(double a, double b, v4 c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int r) { return 4 * r + (l >> 4); }
};

// lane l: A[l % 16][l / 16], B[l / 16][l % 16]; result element r of lane l is
// D[4 (l / 16) + r][l % 16]
template <> struct Mfma<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4 step(float a, float b, v4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int r) { return 4 * (l >> 4) + r; }
};

template <typename R> struct Eps;
template <> struct Eps<double> { static constexpr double v = DBL_EPSILON; };
template <> struct Eps<float> { static constexpr float v = FLT_EPSILON; };

// Sign class of f(t) = a + t (b + t (c + t d)) on [0, h], with the
// evaluation-error margin tol:
// 1 = f >= -tol on the piece: the clipping can only drop values within the
//     rounding margin of zero (pieces that end on a zero knot with zero
//     slope, next to hidden leaves, fall here);
// 0 = f <= tol on the piece, or identically zero;
// 2 = otherwise, evaluated point by point with the clipping.
// The cubic Bernstein coefficients bound f (the curve lies in their convex
// hull) and settle most pieces; the rest are decided by f at the ends and at
// the critical points in (0, h).  The classes 0 and 1 differ from per-point
// clipping by at most tol x area per query, at queries whose value lies
// within tol of zero.
template <typename R>
__device__ __forceinline__ int cubic_class(R a, R b, R c, R d, R h)
{
    if (a == (R)0 && b == (R)0 && c == (R)0 && d == (R)0) return 0;
    const R bh = b * h, ch = c * h * h, dh = d * h * h * h;
    const R scale = fabs(a) + fabs(bh) + fabs(ch) + fabs(dh);
    const R tol = (R)64 * Eps<R>::v * scale;
    const R b0 = a, b1 = a + bh / (R)3, b2 = a + (R)2 * bh / (R)3 + ch / (R)3, b3 = a + bh + ch + dh;
    R lo = fmin(fmin(b0, b1), fmin(b2, b3)), hi = fmax(fmax(b0, b1), fmax(b2, b3));
    if (lo >= -tol) return 1;
    if (hi <= tol) return 0;
    // extremes: the ends and the roots of f'(t) = b + 2 c t + 3 d t^2 in (0, h)
    auto f = [&](R t) { return a + t * (b + t * (c + t * d)); };
    lo = fmin(a, b3);
    hi = fmax(a, b3);
    R r1 = (R)-1, r2 = (R)-1;
    if (d != (R)0) {
        const R disc = c * c - (R)3 * b * d;
        if (disc >= (R)0) {
            const R q = -(c + copysign(sqrt(disc), c));
            if (q != (R)0) { r1 = q / ((R)3 * d); r2 = b / q; }
            else r1 = (R)0;
        }
    } else if (c != (R)0) r1 = -b / ((R)2 * c);
    if (r1 > (R)0 && r1 < h) { const R v = f(r1); lo = fmin(lo, v); hi = fmax(hi, v); }
    if (r2 > (R)0 && r2 < h) { const R v = f(r2); lo = fmin(lo, v); hi = fmax(hi, v); }
    if (lo >= -tol) return 1;
    if (hi <= tol) return 0;
    return 2;
}

}  // namespace xh
