// Compact single-precision sin/cos for the nonlinear phase factors.
//
// Method: Cody-Waite argument reduction by pi/2 with a three-term split of
// pi/2 applied through fused multiply-adds, then Taylor polynomials of sin
// (to r^9) and cos (to r^10) on |r| <= pi/4, whose truncation errors
// (< 3e-9 and < 2e-10) are far below one single-precision ulp.  Every
// operation is an IEEE single-precision fma, multiply, add or round-to-nearest,
// so the host build of this header computes bit-identical results to the
// device build; the unit test checks the host build against double precision.
// Valid for |x| < 2^15 (the reduction constant products stay exact enough).
#pragma once

#include <math.h>
#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__) || defined(__HIP__)
#define BEC_HD __host__ __device__
#else
#define BEC_HD
#endif

namespace bec {

// pi/2 = PIO2_A + PIO2_B + PIO2_C, each the float nearest to the remainder
constexpr float PIO2_A = 1.57079637050628662109375f;
constexpr float PIO2_B = -4.371138828673793e-8f;
constexpr float PIO2_C = -1.7151245100058819e-15f;
constexpr float TWO_OVER_PI = 0.636619746685028076171875f;

BEC_HD inline void fast_sincosf(float x, float *s, float *c)
{
    const float q = rintf(x * TWO_OVER_PI);
    float r = fmaf(-q, PIO2_A, x);
    r = fmaf(-q, PIO2_B, r);
    r = fmaf(-q, PIO2_C, r);
    const float r2 = r * r;
    // sin r = r + r^3 (-1/3! + r^2 (1/5! + r^2 (-1/7! + r^2 / 9!)))
    float ps = fmaf(r2, 2.75573192239858906526e-6f, -1.98412698412698412698e-4f);
    ps = fmaf(r2, ps, 8.33333333333333333333e-3f);
    ps = fmaf(r2, ps, -1.66666666666666666667e-1f);
    const float sn = fmaf(r * r2, ps, r);
    // cos r = 1 + r^2 (-1/2 + r^2 (1/4! + r^2 (-1/6! + r^2 (1/8! - r^2 / 10!))))
    float pc = fmaf(r2, -2.75573192239858906526e-7f, 2.48015873015873015873e-5f);
    pc = fmaf(r2, pc, -1.38888888888888888889e-3f);
    pc = fmaf(r2, pc, 4.16666666666666666667e-2f);
    pc = fmaf(r2, pc, -0.5f);
    const float cs = fmaf(r2, pc, 1.0f);
    const int k = (int)q;
    const bool swap = (k & 1) != 0;
    float ss = swap ? cs : sn;
    float cc = swap ? sn : cs;
    if (k & 2) ss = -ss;
    if ((k + 1) & 2) cc = -cc;
    *s = ss;
    *c = cc;
}

// pi = PI_A + PI_B + PI_C, each the float nearest to the remainder
constexpr float PI_A = 3.1415927410125732421875f;
constexpr float PI_B = -8.742277657347586e-8f;
constexpr float PI_C = -3.4302490200117637e-15f;
constexpr float INV_PI = 0.3183098733425140380859375f;

BEC_HD inline float xor_bits(float v, unsigned m)
{
    unsigned u;
    memcpy(&u, &v, sizeof(u));
    u ^= m;
    memcpy(&v, &u, sizeof(v));
    return v;
}

// Adding 1.5 * 2^23 to |v| < 2^22 rounds v to an integer held in the sum's low
// mantissa bits (the sum lies in [2^23, 2^24), where one ulp is 1).
constexpr float ROUND_MAGIC = 12582912.0f;

// The same accuracy for |x| < 1e5 with a reduction by pi instead of pi/2: x = q pi + r,
// |r| <= pi/2, sin x = (-1)^q sin r and cos x = (-1)^q cos r, so the quadrant
// fix-up is one sign-bit xor per result instead of a swap and two selects.
// Taylor polynomials of sin to r^13 and cos to r^14 (truncation errors
// < 7e-10 and < 7e-11 at pi/2).
//
// Both results come out multiplied by S, which must be a power of two (1 for
// the plain functions): every coefficient and the reduced argument are scaled
// by S before they enter the fused multiply-adds, and scaling by a power of two
// commutes with rounding (no overflow or underflow occurs here), so the results
// are exactly S sin x and S cos x as the unscaled evaluation rounds them.  A
// caller that multiplies sin and cos by a constant power of two anyway (the
// 1/N^2 of an unnormalised transform pair) gets that product for one multiply
// instead of two.  The quadrant q comes from one fused multiply-add with
// ROUND_MAGIC; its parity is the low bit of that sum.
BEC_HD inline void fast_sincos_pi_scaled(float x, float S, float *s, float *c)
{
    const float t = fmaf(x, INV_PI, ROUND_MAGIC);
    const float q = t - ROUND_MAGIC;
    float r = fmaf(-q, PI_A, x);
    r = fmaf(-q, PI_B, r);      // the PI_C term, |q| 3.4e-15, is below 1e-10 for |x| < 1e5
    const float r2 = r * r;
    float ps = fmaf(r2, S * 1.6059043836821614599e-10f, S * -2.5052108385441718775e-8f);
    ps = fmaf(r2, ps, S * 2.7557319223985890653e-6f);
    ps = fmaf(r2, ps, S * -1.9841269841269841270e-4f);
    ps = fmaf(r2, ps, S * 8.3333333333333333333e-3f);
    ps = fmaf(r2, ps, S * -1.6666666666666666667e-1f);
    const float sn = fmaf(r * r2, ps, S * r);
    float pc = fmaf(r2, S * -1.1470745597729724714e-11f, S * 2.0876756987868098979e-9f);
    pc = fmaf(r2, pc, S * -2.7557319223985890653e-7f);
    pc = fmaf(r2, pc, S * 2.4801587301587301587e-5f);
    pc = fmaf(r2, pc, S * -1.3888888888888888889e-3f);
    pc = fmaf(r2, pc, S * 4.1666666666666666667e-2f);
    pc = fmaf(r2, pc, S * -0.5f);
    const float cs = fmaf(r2, pc, S);
    unsigned tb;
    memcpy(&tb, &t, sizeof(tb));
    const unsigned sign = tb << 31;
    *s = xor_bits(sn, sign);
    *c = xor_bits(cs, sign);
}

BEC_HD inline void fast_sincos_pi(float x, float *s, float *c)
{
    fast_sincos_pi_scaled(x, 1.0f, s, c);
}

// pi/2 = DPIO2_A + DPIO2_B + DPIO2_C, each the double nearest to the remainder
constexpr double DPIO2_A = 1.57079632679489655800e+00;
constexpr double DPIO2_B = 6.12323399573676603587e-17;
constexpr double DPIO2_C = -1.49738490485916983294e-33;
constexpr double DTWO_OVER_PI = 6.36619772367581382433e-01;
constexpr double DROUND_MAGIC = 6755399441055744.0;   // 1.5 * 2^52, as ROUND_MAGIC
constexpr double DSINCOS_MAX = 1099511627776.0;   // 2^40

// sin and cos of r + tail, |r| <= pi/4 and |tail| below r's rounding: Taylor
// polynomials of sin (to r^19) and cos (to r^18), whose truncation errors are below
// 1e-21 and 3e-21.
BEC_HD inline void sincos_reduced(double r, double tail, double *s, double *c)
{
    const double r2 = r * r;
    double ps = fma(r2, -8.2206352466243297170e-18, 2.8114572543455207632e-15);
    ps = fma(r2, ps, -7.6471637318198164759e-13);
    ps = fma(r2, ps, 1.6059043836821614599e-10);
    ps = fma(r2, ps, -2.5052108385441718775e-8);
    ps = fma(r2, ps, 2.7557319223985890653e-6);
    ps = fma(r2, ps, -1.9841269841269841270e-4);
    ps = fma(r2, ps, 8.3333333333333333333e-3);
    ps = fma(r2, ps, -1.6666666666666666667e-1);
    *s = r + fma(r * r2, ps, tail);
    double pc = fma(r2, -1.5619206968586226462e-16, 4.7794773323873852974e-14);
    pc = fma(r2, pc, -1.1470745597729724714e-11);
    pc = fma(r2, pc, 2.0876756987868098979e-9);
    pc = fma(r2, pc, -2.7557319223985890653e-7);
    pc = fma(r2, pc, 2.4801587301587301587e-5);
    pc = fma(r2, pc, -1.3888888888888888889e-3);
    pc = fma(r2, pc, 4.1666666666666666667e-2);
    // 1 - r^2/2 rounded, and what that rounding lost
    const double hz = 0.5 * r2, w = 1.0 - hz;
    *c = w + (((1.0 - w) - hz) + fma(r2 * r2, pc, -r * tail));
}

// Double-precision sine and cosine for |x| < DSINCOS_MAX, the FP64 counterpart of
// fast_sincosf: x - q DPIO2_A is exact in one fused multiply-add (a multiple of
// min(ulp(x), 2^-52) below one), the second part of pi/2 enters by two more
// that keep the rounding of the reduced argument.  About 45 operations, without the
// branch of the library function to its long reduction.  Beyond DSINCOS_MAX r0 - r is
// no longer exact.
BEC_HD inline void fast_sincos_f64(double x, double *s, double *c)
{
    const double t = fma(x, DTWO_OVER_PI, DROUND_MAGIC);
    const double q = t - DROUND_MAGIC;
    const double r0 = fma(-q, DPIO2_A, x);
    const double r = fma(-q, DPIO2_B, r0);
    const double tail = fma(-q, DPIO2_C, fma(-q, DPIO2_B, r0 - r));   // what r's rounding lost
    double sn, cs;
    sincos_reduced(r, tail, &sn, &cs);
    uint64_t k;   // the quadrant is in the low mantissa bits of t
    memcpy(&k, &t, sizeof(k));
    const bool swap = (k & 1) != 0;
    const double ss = swap ? cs : sn, cc = swap ? sn : cs;
    *s = (k & 2) ? -ss : ss;
    *c = ((k + 1) & 2) ? -cc : cc;
}

// cos and sin of 2 pi m / n for 0 <= m < n < 2^27: the octant from the integers, so
// that only an angle of at most pi/4 is rounded, and that with its tail: each within
// 1.1e-16.  Rounding 2 m / n itself costs up to pi 2^-53 of angle in the second half,
// whose entries then no longer cancel those of the first: a pair of folded DFTs with
// such a table changed the norm of a 63-point line by 1.6e-16, with these by 2.4e-17.
BEC_HD inline void unit_root(int m, int n, double *c, double *s)
{
    const int k = 2 * m > n ? n - m : m;           // the upper half mirrored
    const int oct = 8 * k / n;                     // 0..4
    int r = 8 * k - oct * n;                       // angle = (oct + r / n) pi/4
    if (oct & 1) r = n - r;                        // from the nearer multiple of pi/2
    const double d = 2.0 * n, q = r / d, ql = fma(-q, d, (double)r) / d;
    const double x = DPIO2_A * q, e = fma(DPIO2_A, q, -x) + (DPIO2_B * q + DPIO2_A * ql);
    double sn, cs;
    sincos_reduced(x, e, &sn, &cs);
    if (oct & 1) sn = -sn;
    const int quad = (oct + 1) >> 1;
    *c = quad == 0 ? cs : quad == 1 ? -sn : -cs;
    const double up = quad == 0 ? sn : quad == 1 ? cs : -sn;
    *s = k != m ? -up : up;
}

} // namespace bec
