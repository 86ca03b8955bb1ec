// mathf64.h - FP64 natural logarithm and quotients for the Model B chemical potentials.
//
// The device library's log carries double-double corrections (about 90 VALU
// instructions on gfx950); the potentials take four logarithms per cell, which
// made them the largest single cost of the Model B step. This one follows the
// classical argument reduction
//
//     x = 2^k (1 + f),  sqrt(2)/2 <= 1 + f < sqrt(2),  s = f / (2 + f),
//     log(1 + f) = 2 atanh(s) = 2s + 2s^3/3 + 2s^5/5 + ...
//               = f - s f + s R,   R = s^2 P(s^2),
//
// with |s| <= 0.1716 (s^2 <= 0.0295). P has degree 6, fitted by Remez exchange to
// 2/3 + 2 s^2/5 + 2 s^4/7 + ... with weight s^2 over that range; it leaves a
// relative error of 2^-58.9 (the series itself needs ten terms for 2^-56). With
// hf = f^2 / 2 (f - s f = f - hf + s hf) the result is assembled as
//     a + (b - (hf - (s (hf + R) + k ln2_lo))),  a + b = k ln2_hi + f,
// k ln2_hi exact for |k| < 2^11. The error stays within 1 ulp of the exact
// logarithm (checked against the C library on the host by the tests, where the same
// source compiles as plain C++): on (0, 1) 0.292 ulp rms, 0.83 at most. (The series
// with ten terms, its quotient taken with two Newton steps and its result without
// fused products: 0.303 and 0.84; Model B step, us: 256^3 580 -> 568, conserved
// 224 x 200 x 180 448 -> 414, 96 x 80 x 64 58 -> 55, 2D 700^2 155 -> 153.) Special
// cases follow IEEE log: NaN for x < 0 and NaN input, -inf at +-0, +inf at +inf.
#pragma once
#include <cmath>

#if defined(__HIPCC__)
#define DBA_HD __host__ __device__
#else
#define DBA_HD
#endif

namespace dba {

// f / b for b in [1.7, 2.42], f 0 or of magnitude in [2^-53, 0.42]: on the device
// Newton's step on the hardware reciprocal (good to 2^-23, then 2^-45), and the
// quotient corrected once by its exact remainder: within 2^-35 ulp of the correctly
// rounded one's bound, without the scaling around the compiler's division.
DBA_HD inline double log_quotient(double f, double b) {
#if defined(__HIP_DEVICE_COMPILE__)
    double y = __builtin_amdgcn_rcp(b);
    y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
    const double q = f * y;
    return __builtin_fma(__builtin_fma(-b, q, f), y, q);
#else
    return f / b;
#endif
}

// a / b for a constant b with y = 1 / b rounded to nearest: the product, corrected once by
// its exact remainder. The product alone is up to 1.5 ulp off; this is the quotient
// rounded to nearest (but for quotients within 2^-51 ulp of a tie). Two operations more
// than the product where a division is a dozen. For finite quotients and remainders
// above the subnormals.
DBA_HD inline double quotient(double a, double b, double y) {
    const double q = a * y;
    return std::fma(std::fma(-b, q, a), y, q);
}

// ... and an infinite or NaN quotient as the product gives it.
DBA_HD inline double quotient_any(double a, double b, double y) {
    const double q = a * y, c = std::fma(std::fma(-b, q, a), y, q);
    return std::fabs(q) < INFINITY ? c : q;
}

// A constant of the series. On the device it is put into scalar registers where it
// is used: hoisted out of a loop, the dozen constants take two vector registers
// each and spill.
DBA_HD inline double log_const(double c) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(c));
#endif
    return c;
}

// log x for positive finite x.
DBA_HD inline double log_positive(double x) {
    int k;
    double m = std::frexp(x, &k);  // m in [0.5, 1), exact for subnormal x too
    const int low = m < log_const(0x1.6a09e667f3bcdp-1);  // sqrt(2)/2
    m = std::ldexp(m, low);
    k -= low;
    const double f = m - 1.0;  // exact (Sterbenz)
    const double s = log_quotient(f, 2.0 + f);
    const double z = s * s;
    double r = log_const(0x1.2f056439aa4b4p-3);
    r = std::fma(r, z, log_const(0x1.39a1baa3e54f2p-3));
    r = std::fma(r, z, log_const(0x1.74663ee942c25p-3));
    r = std::fma(r, z, log_const(0x1.c71c520958848p-3));
    r = std::fma(r, z, log_const(0x1.24924941f12b8p-2));
    r = std::fma(r, z, log_const(0x1.999999997fdb7p-2));
    r = std::fma(r, z, log_const(0x1.5555555555592p-1));
    const double hf = 0.5 * f * f;
    const double dk = (double)k;
    // ln 2 = ln2_hi + ln2_lo, ln2_hi with 21 trailing zero bits
    const double ln2_hi = log_const(0x1.62e42fee00000p-1), ln2_lo = log_const(0x1.a39ef35793c76p-33);
    const double a = std::fma(dk, ln2_hi, f), b = f - std::fma(-dk, ln2_hi, a);  // a + b = k ln2_hi + f
    return a + (b - (hf - std::fma(s, std::fma(z, r, hf), dk * ln2_lo)));
}

DBA_HD inline double log_f64(double x) {
    if (x > 0.0 && x < INFINITY) return log_positive(x);
    return x == 0.0 ? -INFINITY : (x == INFINITY ? x : NAN);
}

}  // namespace dba
