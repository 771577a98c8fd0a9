//----------------------------------*-C++-*----------------------------------//
// celeritas_amd: MI355X-native per-step transport loop
//---------------------------------------------------------------------------//
//! \file corecel/Elementary.hh
//! FP64 logarithm and sine/cosine for the step kernels.
//!
//! The charged along-step executes about 20 logarithms and 6 sines or
//! cosines a track, and its waves are bound by the instructions that they
//! issue. The library carries a logarithm as a pair of doubles from start to
//! end (98 vector instructions; 72 here) and reduces any angle up to the
//! largest double, once for the sine and once for the cosine (260 for both;
//! 70 here). Full TestEm3 transport 840 -> 825 ms, graph replay of 333
//! primaries 48.8 -> 47.5 ms.
//!
//! Largest errors on the device in units of the last place, of eight million
//! values a range (library in parentheses): logarithm of (0, 1) 0.599
//! (0.641), of 0.5 to 2 0.602 (0.637), of 10^-300 to 10^300 0.538 (0.607);
//! sine and cosine of -10 to 10 0.727 (0.779). The mean errors are smaller,
//! too. One part is not: just beside sqrt(1/2) and sqrt(2), where the
//! reduction folds, the logarithm's largest error is 0.611 (0.591 in 1.4142
//! to 1.4143) at a mean of 0.251 (0.254).
//!
//! The logarithm's sum has the form that K. C. Ng published with Sun's
//! freely distributable math library (1993), here with the rounding errors
//! of its large terms; the angle's reduction is Cody and Waite's.
//! Coefficients are interpolations in Chebyshev nodes of the series, taken
//! with 60 digits. The same functions compile for the host; angles above
//! 2^20 radians are out of their range (the kernels' stay below 10).
//---------------------------------------------------------------------------//
#pragma once

#include <cmath>
#include <cstdint>
#include <cstring>

#include "Macros.hh"

namespace celeritas_amd
{
namespace elem
{
namespace detail
{
inline constexpr double ln2_hi = 0x1.62e42fefa3000p-1;  //!< 41 bits
inline constexpr double ln2_lo = 2.8235290563031577e-13;

//! f / (2 + f), with the rounding error of the denominator taken off
CELER_FORCEINLINE_FUNCTION double log_ratio(double f)
{
    double const b = 2 + f;
    double const b_lo = (2 - b) + f;
#if CELER_DEVICE_COMPILE
    double y = __builtin_amdgcn_rcp(b);
    y = std::fma(std::fma(-b, y, 1.0), y, y);
    y = std::fma(std::fma(-b, y, 1.0), y, y);
#else
    double const y = 1 / b;
#endif
    double const q = f * y;
    return std::fma(std::fma(-b_lo, q, std::fma(-b, q, f)), y, q);
}

//! x = m 2^k with m in [sqrt(1/2), sqrt(2))
CELER_FORCEINLINE_FUNCTION double split(double x, int* k)
{
#if CELER_DEVICE_COMPILE
    double const m = __builtin_amdgcn_frexp_mant(x);
    int const e = __builtin_amdgcn_frexp_exp(x);
#else
    int e;
    double const m = std::frexp(x, &e);
#endif
    bool const low = m < 0.70710678118654752;
    *k = low ? e - 1 : e;
    return low ? 2 * m : m;
}

/*!
 * Logarithm of (1 + f + c) 2^k for 1 + f in [sqrt(1/2), sqrt(2)) and a
 * correction c of its last places.
 *
 * With s = f / (2 + f), log(1 + f) = 2 atanh(s) = f - f^2/2 + s (f^2/2 + R)
 * with R = s^2 (2/3 + 2/5 s^2 + ...): f is exact, the sum of the large terms
 * is kept with its rounding error, and the errors of s and R enter through a
 * term of a 20th of the result.
 */
CELER_FORCEINLINE_FUNCTION double log_of(double f, double c, int k)
{
    double const s = log_ratio(f);
    double const z = s * s;
    double q = 0x1.0c04595972ab8p-3;
    q = std::fma(q, z, 0x1.0fbe83c2cbcf3p-3);
    q = std::fma(q, z, 0x1.3b1c360763b8ap-3);
    q = std::fma(q, z, 0x1.745cf901605f7p-3);
    q = std::fma(q, z, 0x1.c71c720160b47p-3);
    q = std::fma(q, z, 0x1.2492492476c87p-2);
    q = std::fma(q, z, 0x1.9999999999a38p-2);
    q = std::fma(q, z, 0x1.5555555555555p-1);
    double const half_f = 0.5 * f;
    double const half_sq = half_f * f;
    double const half_sq_lo = std::fma(half_f, f, -half_sq);
    double const kd = static_cast<double>(k);
    double const a = f - half_sq;
    double const b = kd * ln2_hi;
    double const sum = b + a;
    // Rounding errors of the large terms first (|b| >= |a| unless k is zero),
    // so that the series' term is rounded once
    double low = std::fma(kd, ln2_lo, c - half_sq_lo);
    low += ((f - a) - half_sq) + ((b - sum) + a);
    low = std::fma(s, std::fma(z, q, half_sq), low);
    return sum + low;
}

//! Result of log for arguments that are not positive and finite
CELER_FORCEINLINE_FUNCTION double log_special(double x, double result)
{
    result = x < HUGE_VAL ? result : x;  // +inf, NaN
    result = x == 0 ? -HUGE_VAL : result;
    return x < 0 ? std::nan("") : result;
}
}  // namespace detail

//---------------------------------------------------------------------------//
//! Natural logarithm
CELER_FORCEINLINE_FUNCTION double log(double x)
{
    int k;
    double const m = detail::split(x, &k);
    return detail::log_special(x, detail::log_of(m - 1, 0, k));
}

/*!
 * Sine and cosine of an angle of up to 2^20 radians.
 *
 * The nearest multiple of pi/2 is taken off in two parts (Cody and Waite;
 * the first difference is exact), and both series use the remainder and its
 * rounding error, with the rounding error of the square in their first term.
 */
CELER_FORCEINLINE_FUNCTION void sincos(double x, double* sine, double* cosine)
{
    double const n = std::rint(x * 0.6366197723675814);  // 2/pi
    double const first = std::fma(-n, 0x1.921fb54442d18p+0, x);
    double const r = std::fma(-n, 0x1.1a62633145c07p-54, first);
    double const r_lo = std::fma(-n, 0x1.1a62633145c07p-54, first - r);
    double const z = r * r;
    double const z_lo = std::fma(r, r, -z);
    double const half_z = 0.5 * z;
    double const w = 1 - half_z;

    double p = 0x1.5e0b05bff20f2p-33;
    p = std::fma(p, z, -0x1.ae600aca92c64p-26);
    p = std::fma(p, z, 0x1.71de379654304p-19);
    p = std::fma(p, z, -0x1.a01a019e83816p-13);
    p = std::fma(p, z, 0x1.1111111110bb2p-7);
    double const cube = z * r;
    double const small = std::fma(cube * z, p, std::fma(z_lo * r, -0x1.5555555555555p-3, r_lo * w));
    double const s = r + std::fma(cube, -0x1.5555555555555p-3, small);

    double q = -0x1.907d8f29fe831p-37;
    q = std::fma(q, z, 0x1.1eeb68cd22f56p-29);
    q = std::fma(q, z, -0x1.27e4fa17bf139p-22);
    q = std::fma(q, z, 0x1.a01a019f4e9b4p-16);
    q = std::fma(q, z, -0x1.6c16c16c16967p-10);
    q = std::fma(q, z, 0x1.5555555555555p-5);
    double const c = w + (((1 - w) - half_z) + std::fma(z * z, q, std::fma(-0.5, z_lo, -r * r_lo)));

    int const quadrant = static_cast<int>(n);
    bool const swap = quadrant & 1;
    double const a = swap ? c : s;
    double const b = swap ? s : c;
    *sine = quadrant & 2 ? -a : a;
    *cosine = (quadrant + 1) & 2 ? -b : b;
}

//! Sine of an angle of up to 2^20 radians
CELER_FORCEINLINE_FUNCTION double sin(double x)
{
    double s, c;
    sincos(x, &s, &c);
    return s;
}

//! Cosine of an angle of up to 2^20 radians
CELER_FORCEINLINE_FUNCTION double cos(double x)
{
    double s, c;
    sincos(x, &s, &c);
    return c;
}

//---------------------------------------------------------------------------//
}  // namespace elem
}  // namespace celeritas_amd
