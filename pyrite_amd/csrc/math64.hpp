// math64.hpp -- FP64 elementary functions for kernels whose time is their latency.
//
// The library forms are correct in the last bit or so and long: measured on
// gfx950 with one wave, a logarithm takes about 460 cycles (a double-double
// through a division), a division 100, a square root 150, sin 360.  The forms
// below are FP64 throughout, within about one unit in the last place over the
// ranges they state, and branch-free.
#pragma once

#include "hr_common.hpp"

namespace hr {

constexpr double kLn2Hi = 0x1.62e42fee00000p-1;  // ln 2, upper 32 bits (times an exponent: exact)
constexpr double kLn2Lo = 0x1.a39ef35793c76p-33; // ln 2 - kLn2Hi

// 1/x: hardware estimate and two Newton steps.
__device__ __forceinline__ double rcp_nr(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// a/b from r = 1/b: the product and one correction by its exact remainder (P.
// Markstein, IBM J. Res. Dev. 34 (1990) 111), the correctly rounded quotient but for
// rare last-bit ties.
__device__ __forceinline__ double div_by(double a, double b, double r) {
    const double q = a * r;
    return fma(fma(-q, b, a), r, q);
}

// 1/sqrt(x) for x > 0: hardware estimate and two Newton steps.
__device__ __forceinline__ double rsqrt_nr(double x) {
    double r = __builtin_amdgcn_rsq(x);
    const double h = 0.5 * x;
    r = fma(fma(-h * r, r, 0.5), r, r);
    return fma(fma(-h * r, r, 0.5), r, r);
}

// sqrt(x) for x > 0 (a negative or NaN x gives NaN).
__device__ __forceinline__ double sqrt_nr(double x) { return x * rsqrt_nr(x); }

// ln x for finite x > 0 (a NaN stays one): k ln 2 + 2 atanh(s), s = (m - 1)/(m + 1),
// m in [sqrt(1/2), sqrt(2)), the series of atanh to s^23 (|s| <= 0.1716:
// remainder below 1e-18).
__device__ __forceinline__ double ln(double x) {
    double m = __builtin_amdgcn_frexp_mant(x);
    int k = __builtin_amdgcn_frexp_exp(x);
    const bool low = m < 0.70710678118654752;
    m = low ? m + m : m;
    k = low ? k - 1 : k;
    const double f = m - 1.0, d = m + 1.0, r = rcp_nr(d);
    double s = f * r;
    s = fma(fma(-s, d, f), r, s);
    const double z = s * s, z2 = z * z, z4 = z2 * z2;
    const double a0 = fma(z, 2.0 / 5, 2.0 / 3), a1 = fma(z, 2.0 / 9, 2.0 / 7), a2 = fma(z, 2.0 / 13, 2.0 / 11);
    const double a3 = fma(z, 2.0 / 17, 2.0 / 15), a4 = fma(z, 2.0 / 21, 2.0 / 19);
    const double b0 = fma(z2, a1, a0), b1 = fma(z2, a3, a2), b2 = fma(z2, 2.0 / 23, a4);
    const double P = fma(z4, fma(z4, b2, b1), b0);
    const double e = (double)k;
    return fma(e, kLn2Hi, fma(s, 2.0, fma(s * z, P, e * kLn2Lo)));
}

// exp(x) for finite x: 2^k times the Taylor series to r^13 on |r| <= ln(2)/2
// (remainder below 1e-16); far negative arguments underflow to zero.
__device__ __forceinline__ double exp_any(double x) {
    const double k = rint(x * 1.4426950408889634);
    const double r = fma(k, -kLn2Lo, fma(k, -kLn2Hi, x));
    const double r2 = r * r, r4 = r2 * r2;
    const double a0 = fma(r, 1.0 / 6, 0.5), a1 = fma(r, 1.0 / 120, 1.0 / 24), a2 = fma(r, 1.0 / 5040, 1.0 / 720);
    const double a3 = fma(r, 1.0 / 362880, 1.0 / 40320), a4 = fma(r, 1.0 / 39916800, 1.0 / 3628800);
    const double a5 = fma(r, 1.0 / 6227020800.0, 1.0 / 479001600);
    const double b0 = fma(r2, a1, a0), b1 = fma(r2, a3, a2), b2 = fma(r2, a5, a4);
    return ldexp(fma(r2, fma(r4, fma(r4, b2, b1), b0), r) + 1.0, (int)k);
}

// sin and cos of phi in [0, 2 pi]: the quadrant is taken off with pi/2 in two
// parts and both Taylor series run on |x| <= pi/4 (to x^17 and x^18: remainders
// below 1e-16).
__device__ __forceinline__ void sincos_phi(double phi, double &s, double &c) {
    const double q = rint(phi * 0.63661977236758134);
    double x = fma(-q, 0x1.921fb54442d18p+0, phi);
    x = fma(-q, 0x1.1a62633145c07p-54, x);
    const double z = x * x, z2 = z * z, z4 = z2 * z2;
    const double s0 = fma(z, 1.0 / 120, -1.0 / 6), s1 = fma(z, 1.0 / 362880, -1.0 / 5040);
    const double s2 = fma(z, 1.0 / 6227020800.0, -1.0 / 39916800.0);
    const double s3 = fma(z, 1.0 / 355687428096000.0, -1.0 / 1307674368000.0);
    const double c0 = fma(z, 1.0 / 24, -0.5), c1 = fma(z, 1.0 / 40320, -1.0 / 720);
    const double c2 = fma(z, 1.0 / 479001600.0, -1.0 / 3628800.0);
    const double c3 = fma(z, 1.0 / 20922789888000.0, -1.0 / 87178291200.0);
    const double S = fma(z4, fma(z2, s3, s2), fma(z2, s1, s0));
    const double C = fma(z4, fma(z4, -1.0 / 6402373705728000.0, fma(z2, c3, c2)), fma(z2, c1, c0));
    const double sx = fma(x * z, S, x), cx = fma(z, C, 1.0);
    const int n = (int)q & 3;
    const double a = (n & 1) ? cx : sx, b = (n & 1) ? sx : cx;
    s = (n & 2) ? -a : a;
    c = (n == 1 || n == 2) ? -b : b;
}

}  // namespace hr
