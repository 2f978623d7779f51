// FP64 device arithmetic of the pair sums: reciprocal, reciprocal square root
// and the potential's angle, to the last bits without the compiler's
// correctly rounded sequences (a divide and a square root per pair cost more
// than the rest of the pair together).
#pragma once

#include <hip/hip_runtime.h>

namespace ag2 {

// 1/sqrt(x): the hardware estimate (at most 5.3e-8 relative, measured over
// 1e-60 .. 1e60) and one third-order step, y (1 + e/2 + 3 e^2/8) with e = 1 -
// x y^2, which leaves rounding only (2.2e-16).
__device__ __forceinline__ double rsq_full(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = __builtin_fma(-(x * y), y, 1.0);
    return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
}

// 1/x the same way: y (1 + e + e^2), e = 1 - x y.
__device__ __forceinline__ double rcp_full(double x) {
    const double y = __builtin_amdgcn_rcp(x);
    const double e = __builtin_fma(-x, y, 1.0);
    return __builtin_fma(y, __builtin_fma(e, e, e), y);
}

// atan(x) / x in w = x^2 for |x| <= sqrt(2) - 1: Chebyshev interpolation of
// degree 11 on [0, (sqrt 2 - 1)^2] (error 1.3e-18 in exact arithmetic).
__device__ __forceinline__ double atan_poly(double w) {
    double p = -0.017803896394812564;
    p = __builtin_fma(p, w, 0.03796390316111083);
    p = __builtin_fma(p, w, -0.05035049795312439);
    p = __builtin_fma(p, w, 0.05846866752275139);
    p = __builtin_fma(p, w, -0.06662950246036792);
    p = __builtin_fma(p, w, 0.07692045194561481);
    p = __builtin_fma(p, w, -0.09090896801472813);
    p = __builtin_fma(p, w, 0.11111110744657099);
    p = __builtin_fma(p, w, -0.14285714279244968);
    p = __builtin_fma(p, w, 0.19999999999940837);
    p = __builtin_fma(p, w, -0.3333333333333312);
    return __builtin_fma(p, w, 1.0);
}

// The same for |x| <= 1/16: degree 5 on [0, 1/256] (error 1.3e-19).
__device__ __forceinline__ double atan_poly_small(double w) {
    double p = -0.09001325197487176;
    p = __builtin_fma(p, w, 0.11110718199879728);
    p = __builtin_fma(p, w, -0.14285713490572707);
    p = __builtin_fma(p, w, 0.1999999999927232);
    p = __builtin_fma(p, w, -0.3333333333333309);
    return __builtin_fma(p, w, 1.0);
}

// pi/2 - atan(r / e) = atan(e / r) for r, e >= 0 (not both 0), ir = 1 / r, by
// the largest quotient in the wave: up to 1/16 and up to tan(pi/8) the series
// alone (8 and 14 issue slots; most waves of a tree walk or a direct sum);
// else, with a <= b the smaller and larger of r and e, atan(a / b) = pi/4 +
// atan((a - b) / (a + b)) above tan(pi/8), and the complement where r is the
// smaller (42 slots).
__device__ __forceinline__ double softened_angle(double e, double r, double ir) {
    const double u = e * ir;
    if (__any(!(u <= 0.41421356237309503))) {
        const double a = r < e ? r : e, b = r < e ? e : r;
        const bool up = a > 0.41421356237309503 * b;
        const double num = up ? a - b : a, den = up ? a + b : b;
        const double x = num * rcp_full(den);
        const double t = (up ? 0.78539816339744828 : 0.0) + x * atan_poly(x * x);
        return r < e ? 1.5707963267948966 - t : t;
    }
    if (__any(u > 0.0625)) return u * atan_poly(u * u);
    return u * atan_poly_small(u * u);
}

// The same, a lane's value that of its own branch whatever the wave's others
// need: the wave takes every branch that some lane needs.  (The direct sum of
// 16,384 targets takes 27.7 ms with it, 26.6 with the wave's branch; 29.2 with
// one series of 14 slots up to tan(pi/8).)
__device__ __forceinline__ double softened_angle_own(double e, double r, double ir) {
    const double u = e * ir;
    const bool far = u <= 0.41421356237309503, small = u <= 0.0625;
    double t = 0.0;
    if (__any(small)) t = u * atan_poly_small(u * u);
    if (__any(!small)) {
        if (__any(!far)) {
            const double a = r < e ? r : e, b = r < e ? e : r;
            const bool up = !far && a > 0.41421356237309503 * b;
            const double num = up ? a - b : a, den = up ? a + b : b;
            const double x = far ? u : num * rcp_full(den);
            double v = (up ? 0.78539816339744828 : 0.0) + x * atan_poly(x * x);
            v = r < e ? 1.5707963267948966 - v : v;
            t = small ? t : v;
        } else {
            const double v = u * atan_poly(u * u);
            t = small ? t : v;
        }
    }
    return t;
}

}  // namespace ag2
