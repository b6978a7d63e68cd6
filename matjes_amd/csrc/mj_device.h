// Device-side helpers for the LLG hot path on gfx950.
//
// LLG / euler / langevin evaluate the formulas of
// src/solvers/propagator.f90:13-40, src/solvers/solver.f90:157-178 and
// src/dynamics/BTeff_sd.f90:18-45.  The library is compiled without
// floating-point contraction; where products and sums are fused, fma() says
// so, so that every kernel that runs a stage (compiled per Hamiltonian or
// ahead of time, fused or one launch per stage, batched or not) rounds alike
// and gives the same bits.
//
// What bounds the stage kernels is the issue of instructions, two thirds of them
// FP64 (an LLG evaluation and its euler step took about 140 besides the
// neighbour sum; a wavefront's VALU instruction takes four cycles of its SIMD,
// FP64, integer, move or conversion alike: 1.75 to 1.9 ns measured), so
// the per-site algebra is arranged for few of them without giving up
// accuracy: the constant factor dt / (hbar (1 + alpha^2)) is one operand, the
// unit vector and the restored length are increments about 1 where the
// length allows it (mj_unit, mj_restore), and a rotation is formed without
// its axis and angle (dep_rotate).  Which branch a site takes depends on its
// own values only.  Per step against the correctly rounded square roots and
// quotients of the formulas as they stand: Heun, triangular 2048x2048 at 10 K
// 143.6 -> 113.9 us, 1024x1024 44.7 -> 37.6 us; Depondt, square 768x640 at
// 10 K 22.3 -> 16.9 us.  Against quadruple precision the states are 1.3 to 5
// times closer (Heun, 1000 steps at 10 K: rms 1.0e-14, before 4.9e-14), since
// the length is restored with one rounding.
#pragma once
#ifndef __HIPCC_RTC__
#include <hip/hip_runtime.h>

#include "mj_rngmath.h"
#endif
#include <stdint.h>

#define MJ_HBAR 6.58211928e-1  // eV fs (src/fixed-parameters/constant.f90:25)

struct v3 {
    double x, y, z;
};

__device__ __forceinline__ v3 operator+(v3 a, v3 b)
{
    v3 r;
    r.x = a.x + b.x;
    r.y = a.y + b.y;
    r.z = a.z + b.z;
    return r;
}

__device__ __forceinline__ v3 mk3(double x, double y, double z)
{
    v3 r;
    r.x = x;
    r.y = y;
    r.z = z;
    return r;
}

// cross_NM (src/vector_utils/vector.f90:451-465)
__device__ __forceinline__ v3 cross3(v3 a, v3 b)
{
    return mk3(fma(a.y, b.z, -(a.z * b.y)), fma(a.z, b.x, -(a.x * b.z)), fma(a.x, b.y, -(a.y * b.x)));
}

// c + a x b
__device__ __forceinline__ v3 cross3_add(v3 a, v3 b, v3 c)
{
    return mk3(fma(a.y, b.z, fma(-a.z, b.y, c.x)), fma(a.z, b.x, fma(-a.x, b.z, c.y)),
               fma(a.x, b.y, fma(-a.y, b.x, c.z)));
}

// a + k b
__device__ __forceinline__ v3 fma3(double k, v3 b, v3 a)
{
    return mk3(fma(k, b.x, a.x), fma(k, b.y, a.y), fma(k, b.z, a.z));
}

__device__ __forceinline__ double dot3(v3 a, v3 b) { return fma(a.z, b.z, fma(a.y, b.y, a.x * b.x)); }

// Correctly rounded sqrt(x) and 1 / x for the per-site algebra: the
// instruction sequences the compiler emits for sqrt and 1.0 / x in double
// (rsq / rcp seed, then fma corrections: two Newton steps and a final
// correction for 1 / x, a Goldschmidt step and two corrections for sqrt)
// without their range-scaling steps, which change nothing for x in
// [2^-767, 2^766] (sqrt) and [2^-1000, 2^1000] (1 / x): spin lengths, field
// norms and the Cayley denominator lie far inside.  sqrt(0) = 0 is kept.
// Same bits as the library operations there (checked on the device against
// sqrt and 1.0 / x, mj_math_probe); 8 and 3 fewer instructions per call.
__device__ __forceinline__ double mj_sqrt_rn(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y;
    double h = y * 0.5;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    double d = fma(-g, g, x);
    h = fma(h, r, h);
    g = fma(d, h, g);
    d = fma(-g, g, x);
    g = fma(d, h, g);
    return x == 0.0 ? x : g;
}

__device__ __forceinline__ double mj_rcp_rn(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    const double f = fma(-x, r, 1.0);
    return fma(f, r, r);
}

__device__ __forceinline__ double norm3(v3 a) { return mj_sqrt_rn(dot3(a, a)); }

// 1 / x to about an ulp, x in [2^-1000, 2^1000]: the hardware estimate and two
// Newton steps (mj_rcp_rn without its last correction)
__device__ __forceinline__ double mj_rcp(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}

// The unit vector n = m / |m| of normalize (src/vector_utils/vector.f90:76-84:
// m itself where |m| <= 1e-8), with |m|^2 and 1 / |m|^2 for mj_restore.  A
// spin that euler, Cayley or a rotation left at unit length has
// |m|^2 = 1 + e with e of a few ulp: 1 / |m| = 1 - e/2 to 3 e^2 / 8, below
// 2^-54 for |e| <= 2^-27; one instruction instead of a square root and a
// division (28).  Where |m| <= 1e-8, r2 = infinity sends mj_restore to its
// general branch.
struct MjUnit {
    v3 n;
    double x, r2;
};

__device__ __forceinline__ MjUnit mj_unit(v3 m)
{
    MjUnit u;
    u.x = dot3(m, m);
    double r = mj_fma_k(u.x, -0.5, 1.5);
    u.r2 = r * r;
    if (!(fabs(u.x - 1.0) <= 0x1p-27)) {
        const bool ok = u.x > 1.0e-16;
        r = ok ? mj_rcp_rn(mj_sqrt_rn(u.x)) : 1.0;
        u.r2 = ok ? r * r : __builtin_inf();
    }
    u.n = mk3(m.x * r, m.y * r, m.z * r);
    return u;
}

// t |m| / |t| (the last line of euler, solver.f90:172-176; m where
// |t| <= 1e-8), u = mj_unit(m).  With v = (|m|^2 - |t|^2) / |m|^2 the factor
// is (1 - v)^(-1/2) = 1 + v f(v): t + t (v f) rounds once, where a product
// with |m| and a division by |t| round twice beside the errors of both
// lengths, and v = 0 (a spin at rest) returns t itself.  f of degree 6,
// |v| <= 2^-6 (a turn of up to 7 degrees per stage), within 3e-17 in v f; 13
// instructions instead of 51 (two square roots, a reciprocal and three
// corrected quotients).
__device__ __forceinline__ v3 mj_restore(v3 m, MjUnit u, v3 t)
{
    const double y = dot3(t, t);
    const double v = (u.x - y) * u.r2;
    double f = 0.20955191976592094;
    f = mj_fma_k(f, v, 0.22566986332987313);
    f = mj_fma_k(f, v, 0.24609374032347447);
    f = mj_fma_k(f, v, 0.2734374897543061);
    f = mj_fma_k(f, v, 0.3125000000002953);
    f = mj_fma_k(f, v, 0.3750000000003127);
    f = fma(f, v, 0.5);
    v3 o = fma3(f * v, t, t);
    if (!(fabs(v) <= 0x1p-6)) {
        const double tn = mj_sqrt_rn(y);
        const double s = mj_sqrt_rn(u.x) * mj_rcp_rn(tn);
        o = tn > 1.0e-8 ? mk3(t.x * s, t.y * s, t.z * s) : m;
    }
    return o;
}

// D (1 + a^2) = -n x (B + a n x B), n = m / |m|   (propagator.f90:32-40,
// BTeff_sd.f90:38-43); the division by 1 + a^2 is part of the stage's factor
// k = dt / (hbar (1 + a^2))
__device__ __forceinline__ v3 llg_torque(v3 n, v3 B, double alpha)
{
    return cross3(fma3(alpha, cross3(n, B), B), n);
}

// euler (solver.f90:172-176): t = (m + Dint dt/hbar) + DT dt/hbar, m' = t |m| / |t|;
// dint and dth torques (llg_torque), ki and k their factors: k = dt / (hbar (1 + a^2))
__device__ __forceinline__ v3 euler_step(v3 m, MjUnit u, v3 dint, double ki, v3 dth, double k)
{
    return mj_restore(m, u, fma3(k, dth, fma3(ki, dint, m)));
}

__device__ __forceinline__ v3 euler_step0(v3 m, MjUnit u, v3 dint, double k)
{
    return mj_restore(m, u, fma3(k, dint, m));
}

// Implicit-midpoint (Cayley) solve (I + [a]x) x = m - a x m  (SIB, Mentink et
// al. 2010): x = m + 2 g w, w = u + u x a, u = m x a, g = 1 / (1 + |a|^2); the
// midpoint (m + x) / 2 is m + g w
__device__ __forceinline__ v3 cayley_inc(v3 m, v3 a, double &g)
{
    const v3 u = cross3(m, a);
    g = mj_rcp(fma(a.z, a.z, fma(a.y, a.y, fma(a.x, a.x, 1.0))));
    return cross3_add(u, a, u);
}

__device__ __forceinline__ v3 cayley(v3 m, v3 a)
{
    double g;
    const v3 w = cayley_inc(m, a, g);
    return fma3(2.0 * g, w, m);
}

__device__ __forceinline__ v3 cayley_mid(v3 m, v3 a)
{
    double g;
    const v3 w = cayley_inc(m, a, g);
    return fma3(g, w, m);
}

// a = (dt/2) Omega, Omega = -(B + alpha p x B)/((1+alpha^2) hbar); f = -dt / (2 (1+alpha^2) hbar)
__device__ __forceinline__ v3 sib_vec(v3 p, v3 B, double alpha, double f)
{
    const v3 l = fma3(alpha, cross3(p, B), B);
    return mk3(f * l.x, f * l.y, f * l.z);
}

// Depondt's rotation field times 1 + alpha^2: B + alpha n x B, n = m / |m|
__device__ __forceinline__ v3 dep_field(v3 m, v3 B, double alpha) { return fma3(alpha, cross3(mj_unit(m).n, B), B); }

// m rotated by the vector w = k b (k = dt / (hbar (1 + alpha^2)), b from
// dep_field): Rodrigues without the axis and the angle,
//   m' = m + S w x m + C w x (w x m), S = sin th / th, C = (1 - cos th) / th^2,
// both polynomials in z = th^2 = |w|^2 for th <= 1/2 (within 5e-17 and 3e-18):
// 39 instructions, where the normalised axis and a sincos with its range
// reduction took about 200
__device__ __forceinline__ v3 dep_rotate(v3 m, v3 b, double k)
{
    const v3 w = mk3(k * b.x, k * b.y, k * b.z);
    const double z = dot3(w, w);
    double S = -2.4931934029233215e-08, C = -2.0790894217124703e-09;
    S = mj_fma_k(S, z, 2.7556981477681245e-06);
    C = mj_fma_k(C, z, 2.7557077887523167e-07);
    S = mj_fma_k(S, z, -0.00019841269403598734);
    C = mj_fma_k(C, z, -2.4801586988836374e-05);
    S = mj_fma_k(S, z, 0.00833333333307693);
    C = mj_fma_k(C, z, 0.0013888888888705666);
    S = mj_fma_k(S, z, -0.16666666666666116);
    C = mj_fma_k(C, z, -0.041666666666666276);
    S = fma(S, z, 1.0);
    C = fma(C, z, 0.5);
    if (!(z <= 0.25)) {
        const double th = sqrt(z);
        double st, ct;
        sincos(th, &st, &ct);
        S = st / th;
        C = (1.0 - ct) / z;
    }
    const v3 u = cross3(w, m);
    return fma3(C, cross3(w, u), fma3(S, u, m));
}

// energy of a site: m.(H m) + b.(Z m) + m.H_fft = m.(a/2 + z), a the
// neighbour sum, z = Z^T b + H_fft
__device__ __forceinline__ double mj_site_energy(v3 m, v3 a, v3 z)
{
    return dot3(m, fma3(0.5, a, z));
}

// ---------------------------------------------------------------------------
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) and Box-Muller normals.
// Key = seed, counter = (site, step lo, step hi, stream).
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ uint32_t mj_xor3(uint32_t a, uint32_t b, uint32_t c)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);   // one instruction
#else
    return a ^ b ^ c;
#endif
}

__host__ __device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
        uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
        uint32_t n0 = mj_xor3((uint32_t)(p1 >> 32), c[1], k0);
        uint32_t n1 = (uint32_t)p1;
        uint32_t n2 = mj_xor3((uint32_t)(p0 >> 32), c[3], k1);
        uint32_t n3 = (uint32_t)p0;
        c[0] = n0;
        c[1] = n1;
        c[2] = n2;
        c[3] = n3;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

// three N(0,1) for (site, step) from one Philox block, counter (site, step, 0):
// Box-Muller on the 32-bit words, words (0, 1) -> (n0, n1), words (2, 3) -> n2
// (radius from u = (w + 1) 2^-32 in (0, 1], angle 2 pi w 2^-32 in [0, 2 pi);
// mj_rngmath.h's word forms)
__device__ __forceinline__ v3 normals3(uint64_t seed, uint64_t step, uint32_t site)
{
    uint32_t c[4] = {site, (uint32_t)step, (uint32_t)(step >> 32), 0u};
    philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    const double r1 = mj_radius(mj_ln_u32(c[0]));
    const double r2 = mj_radius(mj_ln_u32(c[2]));
    double s1, c1;
    mj_sincos2pi_u32(c[1], &s1, &c1);
    const double c2 = mj_cos2pi_u32(c[3]);
    return mk3(r1 * c1, r1 * s1, r2 * c2);
}
