// normal64.h -- FP64 elementary functions of the step kernels: the Box-Muller
// pair of two Philox words and the sine of a phase in cycles, for the device
// kernels and, unchanged, for a host build that measures their error
// (tests/test_normal64_cpu.py).
//
// The arguments are special, which a general log / sincos cannot use: both
// uniforms are (word + 1/2) 2^-32, so the logarithm needs no range checks and
// the angle reduces exactly in integers, and a field phase is reduced in
// cycles.  A pair costs ~55 FP64 instructions against ~200 of the general
// functions (three transcendentals with their large-argument and special-value
// paths, a correctly rounded square root, two divisions), and these were two
// thirds of an FP64 Heun step: 65,536 particles in a sine field, 4,096 steps,
// 4.72 -> 2.02 ms a pass.  Polynomials are near-minimax fits on the reduced ranges;
// every product that fuses is written as a fused multiply-add under
// `fp contract(off)`, so all kernels form the same bits.
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__)
#define MP_N64 __host__ __device__ inline
#else
#define MP_N64 inline
#endif

namespace mp {

// Reciprocal and reciprocal square root to ~2^-23 (v_rcp_f64, v_rsq_f64); the
// callers refine them.
MP_N64 double rcp_seed(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcp(x);
#else
    return (double)(1.0f / (float)x);
#endif
}

MP_N64 double rsq_seed(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(x);
#else
    return (double)(1.0f / sqrtf((float)x));
#endif
}

MP_N64 double f64fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

// The high word of x, and x with another one.  (Two 32-bit words rather than
// a 64-bit integer: the compiler splits masks of the latter into byte moves.)
#if defined(__HIP_DEVICE_COMPILE__)
typedef uint32_t f64_words __attribute__((ext_vector_type(2)));
MP_N64 uint32_t f64_hi(double x) { return __builtin_bit_cast(f64_words, x).y; }
MP_N64 double f64_with_hi(double x, uint32_t hi)
{
    return __builtin_bit_cast(double, f64_words{__builtin_bit_cast(f64_words, x).x, hi});
}
#else
MP_N64 uint32_t f64_hi(double x)
{
    uint64_t b;
    memcpy(&b, &x, 8);
    return (uint32_t)(b >> 32);
}
MP_N64 double f64_with_hi(double x, uint32_t hi)
{
    uint64_t b;
    memcpy(&b, &x, 8);
    b = (b & 0xffffffffu) | ((uint64_t)hi << 32);
    memcpy(&x, &b, 8);
    return x;
}
#endif

// sqrt of a normal x in about [1e-290, 1e290]: Goldschmidt from the seed
// (2^-45 after one step) and one residual correction, under one ulp.
MP_N64 double sqrt_normal(double x)
{
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
    const double y = rsq_seed(x);
    const double g = x * y, h = 0.5 * y;
    const double g1 = f64fma(g, f64fma(-h, g, 0.5), g);
    return f64fma(f64fma(-g1, g1, x), h, g1);
}

// 1 / sqrt(x) of a normal x, about one ulp: with e = 1 - x y^2 (a seed gives
// |e| < 2^-22), x^-1/2 = y (1 - e)^-1/2 = y (1 + e/2 + 3 e^2/8 + O(2^-67)).
MP_N64 double rsqrt_normal(double x)
{
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
    const double y = rsq_seed(x);
    const double e = f64fma(-(x * y), y, 1.0);
    return f64fma(y * e, f64fma(0.375, e, 0.5), y);
}

// 1 / x of a normal x whose reciprocal is normal, under one ulp
MP_N64 double rcp_normal(double x)
{
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
    const double y = rcp_seed(x);
    const double y1 = f64fma(f64fma(-x, y, 1.0), y, y);
    return f64fma(f64fma(-x, y1, 1.0), y1, y1);
}

// -2 ln((a + 1/2) 2^-32) for a 32-bit a: in [2.3e-10, 45.8].
// x = a + 1/2 = 2^k m with m in [sqrt(1/2), sqrt(2)); ln m = 2 atanh(s) with
// s = (m - 1) / (m + 1), |s| < 0.172, = 2 s + s^3 P(s^2).  For u near 1, k = 32
// and the sum is -4 s alone, so the relative error stays within an ulp.
MP_N64 double minus_two_log_u(uint32_t a)
{
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
    const double x = (double)a + 0.5;
    // the exponent field left after taking sqrt(1/2)'s high word away is k
    const uint32_t hi = f64_hi(x);
    const int32_t k = (int32_t)(hi - 0x3fe6a09eu) >> 20;
    const double m = f64_with_hi(x, hi - ((uint32_t)k << 20));
    const double f = m - 1.0, d = m + 1.0;
    const double y = rcp_seed(d);
    const double r = f64fma(f64fma(-d, y, 1.0), y, y);      // 1/d to ~2^-46
    const double s0 = f * r;
    const double s = f64fma(f64fma(-s0, d, f), r, s0);      // f/d, rounded once more
    const double z = s * s;
    double p = -0x1.2b5f68a50d903p-2;                       // -2 P(z)
    p = f64fma(p, z, -0x1.39fdcceb4bb45p-2);
    p = f64fma(p, z, -0x1.7462b91b8df65p-2);
    p = f64fma(p, z, -0x1.c71c62d5e53e0p-2);
    p = f64fma(p, z, -0x1.2492492dfd86cp-1);
    p = f64fma(p, z, -0x1.9999999995273p-1);
    p = f64fma(p, z, -0x1.5555555555558p+0);
    const double e = (double)(k - 32);
    // ln 2 in two parts, the first short enough that e times it is exact
    const double top = f64fma(e, -0x1.62e42fef00000p+0, -4.0 * s);
    return top + f64fma(e, -0x1.473de6af278edp-33, (s * z) * p);
}

// cos and sin of 2 pi (b + 1/2) 2^-32: quadrant and remainder in integers, so
// the reduced angle t (in quarter turns, |t| <= 1/2) is exact.
MP_N64 void sincos_u(uint32_t b, double &c, double &s)
{
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
    const uint32_t q = (b + 0x20000000u) >> 30;
    const double t = f64fma((double)(int32_t)(b - (q << 30)), 0x1p-30, 0x1p-31);
    const double z = t * t;
    double ps = 0x1.e4a9d9166f052p-25;                      // sin(pi t/2) = t (pi/2 + z Q(z))
    ps = f64fma(ps, z, -0x1.e3027dea82bd7p-19);
    ps = f64fma(ps, z, 0x1.50783208843ebp-13);
    ps = f64fma(ps, z, -0x1.32d2cce500387p-8);
    ps = f64fma(ps, z, 0x1.466bc6775a476p-4);
    ps = f64fma(ps, z, -0x1.4abbce625be52p-1);
    const double sn = f64fma(t, 0x1.921fb54442d18p+0, (t * z) * ps);
    double pc = -0x1.b2f3eb054afcdp-28;                     // cos(pi t/2) = 1 + z C(z)
    pc = f64fma(pc, z, 0x1.f9ce245cada0bp-22);
    pc = f64fma(pc, z, -0x1.a6d1eef479be1p-16);
    pc = f64fma(pc, z, 0x1.e1f5068688d5bp-11);
    pc = f64fma(pc, z, -0x1.55d3c7e3cb241p-6);
    pc = f64fma(pc, z, 0x1.03c1f081b5ac0p-2);
    pc = f64fma(pc, z, -0x1.3bd3cc9be45dep+0);
    const double cn = f64fma(z, pc, 1.0);
    const bool odd = (q & 1u) != 0;
    const double x = odd ? sn : cn, y = odd ? cn : sn;
    c = f64_with_hi(x, f64_hi(x) ^ (((q + 1u) & 2u) << 30));
    s = f64_with_hi(y, f64_hi(y) ^ ((q & 2u) << 30));
}

// The Box-Muller pair of words (a, b): r cos, r sin with r = sqrt(-2 ln u(a)).
MP_N64 void box_muller64(uint32_t a, uint32_t b, double &z0, double &z1)
{
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
    const double r = sqrt_normal(minus_two_log_u(a));
    double c, s;
    sincos_u(b, c, s);
    z0 = r * c;
    z1 = r * s;
}

// sin(2 pi c) for a phase of c cycles, |c| < 2^51: c less its nearest integer
// and the fold about a quarter turn are exact, then t (pi/2 + z Q(z)) with t in
// quarter turns, |t| <= 1.
MP_N64 double sin_cycles(double c)
{
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
    const double r = c - rint(c);
    const double t = 4.0 * (fabs(r) > 0.25 ? copysign(0.5, r) - r : r);
    const double z = t * t;
    double p = 0x1.9ec5cdbeecd34p-38;
    p = f64fma(p, z, -0x1.6f866b70b27bdp-31);
    p = f64fma(p, z, 0x1.e8f3b0121aafdp-25);
    p = f64fma(p, z, -0x1.e3074ee5f4a61p-19);
    p = f64fma(p, z, 0x1.50783486f190cp-13);
    p = f64fma(p, z, -0x1.32d2cce62adb9p-8);
    p = f64fma(p, z, 0x1.466bc6775aad6p-4);
    p = f64fma(p, z, -0x1.4abbce625be53p-1);
    return f64fma(t, 0x1.921fb54442d18p+0, (t * z) * p);
}

}  // namespace mp
