// FP64 ln(u) on (0,1] and (sin, cos)(2 pi u) on [0,1) for the Box-Muller
// thermal field.  Both arguments are uniforms in the unit interval, so the
// general library routines' range handling is not needed:
//   ln u    : u = m 2^e with m in [sqrt(1/2), sqrt(2)), s = (m-1)/(m+1),
//             ln m = 2 atanh(s) = 2s (1 + s^2/3 + s^4/5 + ...) (|s| <= 0.172,
//             series to s^25), ln 2 split hi/lo (the fdlibm constants);
//   sincos  : 8u = octant + f exactly, angle (pi/4) f or (pi/4)(1-f) in
//             [0, pi/4], Taylor series to t^17 / t^18, octant symmetries.
// Accuracy (checked against libm on the host, tests/test_rngmath.py): a few
// ulp.  Plain C++ so the same source compiles for the host test.
//
// The thermal normals use the word forms below (mj_ln_u32, mj_sincos2pi_u32,
// mj_cos2pi_u32, mj_radius): the uniform is taken from its 32-bit word by
// integer operations (octant, fraction and signs of the angle, exponent and
// mantissa of the logarithm: fewer instructions than the FP64 ones they replace;
// each takes the same issue slot),
// the polynomials are the interpolants at Chebyshev nodes of the ranges they
// cover (within 5e-18 to 3e-17, two terms shorter than the series), the
// logarithm's quotient and the square root start from the hardware reciprocal
// / reciprocal square root with fma corrections on the device (IEEE on the
// host), and the third normal needs a cosine only (one sine polynomial on
// [0, pi/2]).  Accuracy: a few ulp (host: tests of these functions against
// libm; device: the normals against the oracle's libm ones).
#pragma once
#include <stdint.h>
#ifndef MJ_HD
#if defined(__HIPCC_RTC__)
#define MJ_HD __host__ __device__ __forceinline__
#elif defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define MJ_HD __host__ __device__ __forceinline__
#else
#define MJ_HD static inline
#include <math.h>
#endif
#endif

// a b + c for a constant c.  On the device c comes from scalar registers: left
// to itself the compiler copies such a constant into vector registers before
// every fma that accumulates onto it, one more issue slot per term of a
// polynomial.  a and b must not be results of v_rcp/v_rsq taken directly (the
// compiler does not insert the wait state those need before inline assembly).
MJ_HD double mj_fma_k(double a, double b, double c)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
    return r;
#else
    return fma(a, b, c);
#endif
}

MJ_HD double mj_log01(double u)
{
    int e;
    double m = frexp(u, &e);                 // u = m 2^e, m in [0.5, 1)
    if (m < 0.70710678118654752440) {
        m = 2.0 * m;
        e = e - 1;
    }
    const double s = (m - 1.0) / (m + 1.0); // m - 1 exact
    const double z = s * s;
    double p = 1.0 / 25.0;
    p = fma(p, z, 1.0 / 23.0);
    p = fma(p, z, 1.0 / 21.0);
    p = fma(p, z, 1.0 / 19.0);
    p = fma(p, z, 1.0 / 17.0);
    p = fma(p, z, 1.0 / 15.0);
    p = fma(p, z, 1.0 / 13.0);
    p = fma(p, z, 1.0 / 11.0);
    p = fma(p, z, 1.0 / 9.0);
    p = fma(p, z, 1.0 / 7.0);
    p = fma(p, z, 1.0 / 5.0);
    p = fma(p, z, 1.0 / 3.0);
    const double s2 = 2.0 * s;
    const double lm = fma(s2, z * p, s2);
    const double de = (double)e;
    return fma(de, 6.93147180369123816490e-01, fma(de, 1.90821492927058770002e-10, lm));
}

MJ_HD void mj_sincos2pi(double u, double *sn, double *cs)
{
    const double x8 = 8.0 * u;               // exact
    const double q = floor(x8);
    const double f = x8 - q;                 // exact, [0, 1)
    const int o = (int)q & 7;
    const double g = (o & 1) ? (1.0 - f) : f;
    const double t = g * 0.78539816339744830962;   // pi/4
    const double t2 = t * t;
    double ps = -1.0 / 355687428096000.0;    // -1/17!
    ps = fma(ps, t2, 1.0 / 1307674368000.0);
    ps = fma(ps, t2, -1.0 / 6227020800.0);
    ps = fma(ps, t2, 1.0 / 39916800.0);
    ps = fma(ps, t2, -1.0 / 362880.0);
    ps = fma(ps, t2, 1.0 / 5040.0);
    ps = fma(ps, t2, -1.0 / 120.0);
    ps = fma(ps, t2, 1.0 / 6.0);
    // sin t = t - t^3 (1/6 - t^2/120 + ...)
    const double st = fma(-(t * t2), ps, t);
    double pc = 1.0 / 6402373705728000.0;    // 1/18!
    pc = fma(pc, t2, -1.0 / 20922789888000.0);
    pc = fma(pc, t2, 1.0 / 87178291200.0);
    pc = fma(pc, t2, -1.0 / 479001600.0);
    pc = fma(pc, t2, 1.0 / 3628800.0);
    pc = fma(pc, t2, -1.0 / 40320.0);
    pc = fma(pc, t2, 1.0 / 720.0);
    pc = fma(pc, t2, -1.0 / 24.0);
    pc = fma(pc, t2, 0.5);
    // cos t = 1 - t^2 (1/2 - t^2/24 + ...)
    const double ct = fma(-t2, pc, 1.0);
    const int swap = ((o + 1) >> 1) & 1;
    const double sa = swap ? ct : st;
    const double ca = swap ? st : ct;
    *sn = (o >= 4) ? -sa : sa;
    *cs = (((o + 2) >> 2) & 1) ? -ca : ca;
}

// a / b for b in [1.7, 2.5] (the logarithm's quotient): on the device the
// hardware reciprocal, one Newton step and one quotient correction (~0.5 ulp)
MJ_HD double mj_div_log(double a, double b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double r = __builtin_amdgcn_rcp(b);
    const double e = fma(-b, r, 1.0);
    r = fma(r, e, r);
    const double q = a * r;
    const double d = fma(-b, q, a);
    return fma(d, r, q);
#else
    return a / b;
#endif
}

// sqrt(-2 l), the Box-Muller radius of l = ln u in [-23, 0]: the hardware
// reciprocal square root, a Goldschmidt step and one correction on the device,
// where 1e-300 stands for 0 (no test for it)
MJ_HD double mj_radius(double l)
{
#if defined(__HIP_DEVICE_COMPILE__)
    const double y = fma(-2.0, l, 1.0e-300);
    const double z = __builtin_amdgcn_rsq(y);
    double g = y * z;
    double h = z * 0.5;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    const double d = fma(-g, g, y);
    return fma(d, h, g);
#else
    return sqrt(-2.0 * l);
#endif
}

// ln((w + 1) 2^-32): x = w + 1 = m 2^e exactly, m in [sqrt(1/2), sqrt(2)] (split
// at the high word of sqrt(1/2)), ln x = e ln 2 + 2 atanh(s), s = (m - 1)/(m + 1),
// |s| <= 0.172
MJ_HD double mj_ln_u32(uint32_t w)
{
    const double x = (double)w + 1.0;
    uint64_t b;
    __builtin_memcpy(&b, &x, sizeof b);
    const uint32_t hi = (uint32_t)(b >> 32);
    const int e = (int)(hi - 0x3FE6A09Eu) >> 20;
    b = (uint64_t)(hi - ((uint32_t)e << 20)) << 32 | (uint32_t)b;
    double m;
    __builtin_memcpy(&m, &b, sizeof m);
    const double s = mj_div_log(m - 1.0, m + 1.0);
    const double z = s * s;
    double p = 0.07308292712444311;
    p = mj_fma_k(p, z, 0.07665855309105386);
    p = mj_fma_k(p, z, 0.09091444727837474);
    p = mj_fma_k(p, z, 0.11111105565129939);
    p = mj_fma_k(p, z, 0.14285714313001635);
    p = mj_fma_k(p, z, 0.19999999999949722);
    p = mj_fma_k(p, z, 0.3333333333333335);
    const double s2 = s + s;
    const double lm = fma(s2, z * p, s2);
    const double de = (double)(e - 32);
    return fma(de, 6.93147180369123816490e-01, fma(de, 1.90821492927058770002e-10, lm));
}

// x with the sign bit flipped where bit 31 of f is set
MJ_HD double mj_flip(double x, uint32_t f)
{
    uint64_t b;
    __builtin_memcpy(&b, &x, sizeof b);
    b ^= (uint64_t)(f & 0x80000000u) << 32;
    __builtin_memcpy(&x, &b, sizeof x);
    return x;
}

// (sin, cos)(2 pi w 2^-32): octant = top 3 bits, v = the distance in 2^-32 of
// the angle from the nearest multiple of pi/2, t = 2 pi v 2^-32 in [0, pi/4]
MJ_HD void mj_sincos2pi_u32(uint32_t w, double *sn, double *cs)
{
    const uint32_t x = w & 0x3FFFFFFFu, x1 = 0x40000000u - x;
    const double t = (double)(x < x1 ? x : x1) * 1.4629180792671596e-09;   // 2 pi 2^-32
    const double t2 = t * t;
    double ps = -1.5918129294866608e-10;
    ps = mj_fma_k(ps, t2, 2.5051131845003624e-08);
    ps = mj_fma_k(ps, t2, -2.755731610255244e-06);
    ps = mj_fma_k(ps, t2, 0.00019841269836758574);
    ps = mj_fma_k(ps, t2, -0.008333333333330948);
    ps = mj_fma_k(ps, t2, 0.16666666666666666);
    const double st = fma(-(t * t2), ps, t);
    double pc = 1.1367998654022494e-11;
    pc = mj_fma_k(pc, t2, -2.0875886738047052e-09);
    pc = mj_fma_k(pc, t2, 2.7557315566341895e-07);
    pc = mj_fma_k(pc, t2, -2.480158729369346e-05);
    pc = mj_fma_k(pc, t2, 0.0013888888888880775);
    pc = mj_fma_k(pc, t2, -0.04166666666666664);
    pc = fma(pc, t2, 0.5);
    const double ct = fma(-t2, pc, 1.0);
    const bool swap = ((w ^ (w >> 1)) & 0x20000000u) != 0;   // octants 1, 2, 5, 6
    *sn = mj_flip(swap ? ct : st, w);
    *cs = mj_flip(swap ? st : ct, w ^ (w << 1));
}

// cos(2 pi w 2^-32) alone: +-sin t, t the angle's distance from the nearest odd
// multiple of pi/2, one sine polynomial on [0, pi/2]; negative in quadrants 1, 2
MJ_HD double mj_cos2pi_u32(uint32_t w)
{
    const uint32_t x = w & 0x3FFFFFFFu;
    const double t = (double)((w & 0x40000000u) ? x : 0x40000000u - x) * 1.4629180792671596e-09;
    const double t2 = t * t;
    double p = -2.7314447669863995e-15;
    p = mj_fma_k(p, t2, 7.643970296798572e-13);
    p = mj_fma_k(p, t2, -1.6058977312464087e-10);
    p = mj_fma_k(p, t2, 2.5052107616996182e-08);
    p = mj_fma_k(p, t2, -2.7557319219163234e-06);
    p = mj_fma_k(p, t2, 0.00019841269841254974);
    p = mj_fma_k(p, t2, -0.008333333333333316);
    p = mj_fma_k(p, t2, 0.16666666666666666);
    return mj_flip(fma(-(t * t2), p, t), w ^ (w << 1));
}
