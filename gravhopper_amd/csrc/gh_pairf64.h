// The FP64 pair factor (1/d)/sqrt(d) of the direct sum, bit for bit as three correctly
// rounded IEEE operations give it (gravhopper/_jbgrav.c:167, :331), from one reciprocal
// square root.  Host and device compile the same function; tests/host/pair_factor_check.cpp
// compares it with the host's division and square root.
//
// What bounds the FP64 direct sum is the FP64 issue rate.  The compiler's expansions of the
// two divisions and the square root take 38 FP64 instructions, three transcendentals (a
// quarter of the rate) and the selects for subnormal, infinite and NaN operands.  The form
// below takes 20 and one transcendental: the square root's iteration also yields the
// reciprocals both divisions need, and operands are restricted to a range where nothing
// underflows or overflows (the caller takes the plain expressions outside).
#pragma once

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)
#define GH_HD __host__ __device__ __forceinline__
#else
#define GH_HD static inline
#endif

namespace gh {

// d is in range when the high word of its bits is in [kPairLoHi, kPairLoHi + kPairSpan),
// 2^-500 <= d < 2^501, and its low word is not all ones.  Then 1/d, sqrt(d) and d^(-3/2)
// and every residual below are normal numbers; zero, negative, subnormal, infinite and NaN
// d are out of range.  (A mantissa of all ones is the one a Newton step rounds 1/d wrongly
// for: 1/d lies 2^-106 above a midpoint and the step lands on it.  Testing the low word
// alone costs one instruction and sends one d in 2^32 to the plain expressions.)
constexpr uint32_t kPairLoHi = (uint32_t)(1023 - 500) << 20;
constexpr uint32_t kPairSpan = (uint32_t)1001 << 20;
constexpr uint32_t kPairLowOnes = 0xffffffffu;

// y0 approximates 1/sqrt(d) to a relative 2^-20 or better (v_rsq_f64: 2^-24.6).
//
// sqrt: Goldschmidt's coupled iteration takes g to sqrt(d) and h to 1/(2 sqrt(d)), both
// to about 2^-48 after one step; two residual corrections g += (d - g^2) h follow, the
// residual exact in one fma.  This is the arithmetic of the compiler's own expansion (its
// scaling is by powers of 4 and does nothing in range), so s is the same bits.
//
// Reciprocals: a Newton step y += y (1 - b y) on a y with relative error e leaves
// (1 - e^2)/b before its rounding (Markstein, IBM J. Res. Dev. 34, 1990).  With b's
// mantissa B and M a midpoint of two neighbouring doubles (54 bits), B M is an integer
// other than a power of two, so 1/b is at least 2^-106 of itself away from any midpoint,
// and with y one of the two doubles around 1/b, e^2 is below that distance unless b's
// mantissa is all ones: the result is the correctly rounded 1/b.  A step on any y with
// e < 2^-30 gives one of those two doubles.  a (for 1/d) starts at 2^-50 and takes both steps, so a is 1.0 / d.  y (for
// 1/s) starts at 2^-48 and takes one: |y - 1/s| is at most half an ulp and 2^-95.
//
// Quotient: q = a y is within 1.3 ulp of a/s, its residual r is exact whenever a/s is near
// a midpoint, and q + r y before rounding is off by at most (half an ulp of q) x s x
// |y - 1/s|.  a/s is at least (quarter ulp of q) x 2^-52 / s from a midpoint, which is
// larger unless s is within 2^-42 of the next power of two; there only d with a/s within
// 2^-53 ulp of a midpoint could round differently, and the host check runs every d whose
// root is that close.
GH_HD double pair_factor(double d, double y0)
{
    double g = d * y0, h = 0.5 * y0;
    double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    r = fma(-g, g, d);
    g = fma(r, h, g);
    r = fma(-g, g, d);
    const double s = fma(r, h, g);
    double y = h + h;
    double e = fma(-s, y, 1.0);
    y = fma(e, y, y);
    double a = y * y;
    e = fma(-d, a, 1.0);
    a = fma(e, a, a);
    e = fma(-d, a, 1.0);
    a = fma(e, a, a);
    const double q = a * y;
    r = fma(-s, q, a);
    return fma(r, y, q);
}

}  // namespace gh
