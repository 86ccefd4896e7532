// Near-field kernel arithmetic: e^{ikr}/r (and the field weight) from an FP64 r^2, in FP32 for
// mixed plans and in FP64 for FP64 plans and the direct sum.  Compiled for the GPU by hipcc
// and for the host by g++ (the host build is how the error bounds of these functions are
// tested without a GPU); the only difference is the reciprocal square root: the GPU's
// v_rsq_f32 (about 1 ulp) on the device, 1/sqrtf on the host (correctly rounded square root,
// then a correctly rounded division), and in FP64 the estimate that both refine.
#pragma once

#include <cmath>
#include <cstdint>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define HFMM_HD __host__ __device__
#else
#define HFMM_HD
#endif

namespace hfmm {
namespace nearfield {

HFMM_HD inline uint32_t fbits(float x) { return __builtin_bit_cast(uint32_t, x); }
HFMM_HD inline float bitsf(uint32_t x) { return __builtin_bit_cast(float, x); }
HFMM_HD inline uint64_t dbits(double x) { return __builtin_bit_cast(uint64_t, x); }

HFMM_HD inline float rsq(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsqf(x);
#else
    return 1.0f / std::sqrt(x);
#endif
}

// ---------------------------------------------------------------------------------
// Half-turn form.  With u = k r / pi, e^{ikr} = e^{i pi u} = (-1)^n e^{i pi y}, where
// n = rint(u) and y = u - n lies in [-1/2, 1/2].  rint comes from adding 1.5 * 2^23
// (1.5 * 2^52 in FP64): the sum is an integer in binary32 whose last mantissa bit is the
// parity of n, and that bit becomes the sign of 1/u with one shift-or (1/u > 0, so OR is
// XOR).  Callers stage coordinates multiplied by k / pi, so u comes from r^2 directly and
// the potential is the sum of these weights times k / pi.
// ---------------------------------------------------------------------------------

// sin(pi y) and cos(pi y) for |y| <= 1/2: minimax polynomials (Remez, absolute error) of
// degree 9 (odd) and 10 (even) with binary32 coefficients, generated by
// hfmm0_amd/csrc/sincos_remez.py; approximation error 4.9e-8 (sin) and 1.8e-8 (cos).
HFMM_HD inline void sincospi_half(float y, float& s, float& c) {
    const float t = y * y;
    float ps = fmaf(t, 7.722012699e-02f, -5.980451703e-01f);
    ps = fmaf(t, ps, 2.550031424e+00f);
    ps = fmaf(t, ps, -5.167706966e+00f);
    ps = fmaf(t, ps, 3.141592503e+00f);
    s = y * ps;
    float pc = fmaf(t, -2.439671569e-02f, 2.349375635e-01f);
    pc = fmaf(t, pc, -1.335212111e+00f);
    pc = fmaf(t, pc, 4.058709145e+00f);
    pc = fmaf(t, pc, -4.934802055e+00f);
    c = fmaf(t, pc, 1.0f);
}

// e^{i pi u} / u from u2 = u^2 > 0 (binary32 normal), all in FP32, as cos(pi y), sin(pi y)
// and the signed 1/u: the weight is (c rs, s rs).  The phase carries the rounding of u,
// about u 2^-24 rad: the form for pairs with moderate k r.
HFMM_HD inline void halfturn_parts(float u2, float& c, float& s, float& rs) {
    const float rinv = rsq(u2);
    const float u = u2 * rinv;
    const float m = u + 12582912.0f;          // 1.5 * 2^23
    const float n = m - 12582912.0f;
    const float y = u - n;
    sincospi_half(y, s, c);
    rs = bitsf((fbits(m) << 31) | fbits(rinv));
}

// The same with u and its reduction in FP64 (u from the FP32 estimate u2 rsq(u2) and one
// Newton step, relative error ~1e-14): the phase stays accurate to FP64 rounding for
// pairs reaching large k r; sin and cos of the reduced y are the FP32 polynomials.
HFMM_HD inline void halfturn_parts_phase64(double u2, float& c, float& s, float& rs) {
    const float u2f = (float)u2;
    const float rinv = rsq(u2f);
    const double u0 = (double)(u2f * rinv);
    const double u = fma((double)(0.5f * rinv), fma(-u0, u0, u2), u0);
    const double m = u + 6755399441055744.0;  // 1.5 * 2^52
    const double n = m - 6755399441055744.0;
    const float y = (float)(u - n);
    sincospi_half(y, s, c);
    rs = bitsf(((uint32_t)dbits(m) << 31) | fbits(rinv));
}

HFMM_HD inline void halfturn_weight(float u2, float& wr, float& wi) {
    float c, s, rs;
    halfturn_parts(u2, c, s, rs);
    wr = c * rs;
    wi = s * rs;
}

HFMM_HD inline void halfturn_weight_phase64(double u2, float& wr, float& wi) {
    float c, s, rs;
    halfturn_parts_phase64(u2, c, s, rs);
    wr = c * rs;
    wi = s * rs;
}

// Weight of one pair of the mixed near field from the scaled r^2 (FP64): e^{i pi u}/u, and
// zero at or below the floor fl2 (fl2 >= 2^-120).  r^2 is raised to at least 2^-120 before
// the arithmetic, so c and s stay finite at r = 0 and the zeroed rs gives exact zeros.
template <bool PH>
HFMM_HD inline void pair_weight(double r2, double fl2, float& wr, float& wi) {
    const bool ok = r2 > fl2;
    float c, s, rs;
    if constexpr (PH)
        halfturn_parts_phase64(fmax(r2, 0x1p-120), c, s, rs);
    else
        halfturn_parts(fmaxf((float)r2, 0x1p-120f), c, s, rs);
    rs = ok ? rs : 0.0f;
    wr = c * rs;
    wi = s * rs;
}

// ---------------------------------------------------------------------------------
// FP64 half-turn form (FP64 plans and the direct sum).
// ---------------------------------------------------------------------------------

// k / pi as an unevaluated sum of two FP64 values (relative error about 2^-105)
struct HalfTurnK {
    double hi, lo;
};
inline HalfTurnK halfturn_k(double k) {
    const double pi_hi = 3.1415926535897931160, pi_lo = 1.2246467991473532072e-16;
    const double hi = k / pi_hi;
    return HalfTurnK{hi, (std::fma(-hi, pi_hi, k) - hi * pi_lo) / pi_hi};
}

// an estimate of x^-1/2 with relative error below 1e-6 (v_rsq_f64: measured 5.2e-8)
HFMM_HD inline double rsq64_estimate(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(x);
#else
    return (1.0 / std::sqrt(x)) * (1.0 - 6e-8);   // the device's error, so that host tests see the correction work
#endif
}

// 1/r and r from r2 = r^2 > 0.  With y the estimate and e = 1 - r2 y^2,
// r^-1 = y (1 - e)^-1/2 = y (1 + e/2 + 3 e^2/8) up to 5 e^3 / 16 (e <= 2e-6: below 1e-17); r is
// r2 / r with one correction from its residual.  A subnormal r2 holds fewer bits, which the residual
// of r then rounds to as well; 1/r is that of the r2 given.
HFMM_HD inline void rsqrt64(double r2, double& rinv, double& r) {
    const double y = rsq64_estimate(r2);
    const double e = fma(-(r2 * y), y, 1.0);
    rinv = fma(y * e, fma(e, 0.375, 0.5), y);
    const double t = r2 * rinv;
    r = fma(0.5 * rinv, fma(-t, t, r2), t);
}

// sin(pi y) and cos(pi y) for |y| <= 1/2: minimax polynomials (Remez, absolute error) of
// degree 17 (odd) and 16 (even), generated by hfmm0_amd/csrc/sincos_remez.py;
// approximation error with the binary64 coefficients 5.4e-17 (sin) and 1.2e-16 (cos).
// The kernels hold the coefficients in scalar registers (`pinned`): FP64 FMAs take a scalar
// addend, while the compiler left to itself keeps them in vector registers and copies one
// before every step, since its accumulating FMA overwrites the addend.
struct SinCosPi64 {
    double s[9] = {3.14159265358979312e+00,  -5.16771278004996848e+00, 2.55016403987724116e+00,
                   -5.99264529317457884e-01, 8.21458865532826710e-02,  -7.37043035602404084e-03,
                   4.66299170571231986e-04,  -2.19020215213132668e-05, 7.68394041277779699e-07};
    double c[9] = {1.0,
                   -4.93480220054467633e+00, 4.05871212641649759e+00, -1.33526276884346462e+00,
                   2.35330630129808288e-01,  -2.58068887393525410e-02, 1.92955628359191256e-03,
                   -1.04566580734636122e-04, 4.14959170019500732e-06};
    HFMM_HD static inline SinCosPi64 pinned() {
        SinCosPi64 p;
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
        for (int i = 0; i < 9; ++i) asm("" : "+s"(p.s[i]));
#pragma unroll
        for (int i = 1; i < 9; ++i) asm("" : "+s"(p.c[i]));
#endif
        return p;
    }
};

HFMM_HD inline void sincospi_half64(double y, const SinCosPi64& p, double& s, double& c) {
    const double t = y * y;
    double ps = fma(t, p.s[8], p.s[7]), pc = fma(t, p.c[8], p.c[7]);
#pragma unroll
    for (int i = 6; i >= 0; --i) {
        ps = fma(t, ps, p.s[i]);
        pc = fma(t, pc, p.c[i]);
    }
    s = y * ps;
    c = pc;
}

// e^{ikr} = (-1)^n (c + i s) from r2 = r^2 > 0 in FP64: c = cos(pi y), s = sin(pi y), and rs
// the signed 1/r, so that e^{ikr}/r is (c rs, s rs); also 1/r and r.  The reduction
// y = r k/pi - n takes k/pi in two terms, so only its own rounding (2^-53 of n) and r's enter
// the phase.  r^2 = 0 counts as the smallest subnormal number (1/r^2 overflows there).  Beyond
// k r / pi = 2^50, where an FP64 k r carries an error of a radian, the phase stays that of
// 2^50 (the parity trick needs integers below 2^51).
HFMM_HD inline void halfturn64(double r2, HalfTurnK k, const SinCosPi64& sp, double& c, double& s, double& rs, double& rinv, double& r) {
    rsqrt64(fmax(r2, 0x1p-1074), rinv, r);
    const double p = fmin(r * k.hi, 0x1p50);
    const double m = p + 6755399441055744.0;  // 1.5 * 2^52
    const double n = m - 6755399441055744.0;
    const double y = fmin(fma(r, k.lo, fma(r, k.hi, -n)), 0.5);
    sincospi_half64(y, sp, s, c);
    rs = __builtin_bit_cast(double, dbits(rinv) | (dbits(m) << 63));
}

// Weight of one pair in FP64, e^{ikr}/r, exactly zero at or below the floor fl2.  A pair at the
// floor contributes nothing whatever its charge: with a charge that is not finite the caller leaves
// the pair out, 0 x NaN being NaN.
HFMM_HD inline void pair_weight64(double r2, double fl2, HalfTurnK k, const SinCosPi64& sp, double& wr,
                                  double& wi) {
    double c, s, rs, rinv, r;
    halfturn64(r2, k, sp, c, s, rs, rinv, r);
    rs = r2 > fl2 ? rs : 0.0;
    wr = c * rs;
    wi = s * rs;
}

// false for every charge that is not finite (and for finite ones whose parts' sum overflows)
HFMM_HD inline bool finite_charge(double re, double im) { return fabs(re) + fabs(im) < __builtin_inf(); }

// ---------------------------------------------------------------------------------
// Radian form (the field kernel): y = k r reduced by pi to [-pi/2, pi/2].
// ---------------------------------------------------------------------------------

// sin and cos in FP32 of y in [-pi/2, pi/2]: the Taylor polynomials of degree 13 (sin) and
// 14 (cos), whose truncation errors on that interval are below 6.6e-10 and 6.5e-11.
HFMM_HD inline void sincos_halfpi(float y, float& s, float& c) {
    const float y2 = y * y;
    float ps = fmaf(y2, 1.6059043836821615e-10f, -2.5052108385441719e-8f);
    ps = fmaf(y2, ps, 2.7557319223985893e-6f);
    ps = fmaf(y2, ps, -1.9841269841269841e-4f);
    ps = fmaf(y2, ps, 8.3333333333333333e-3f);
    ps = fmaf(y2, ps, -1.6666666666666667e-1f);
    s = fmaf(y * y2, ps, y);
    float pc = fmaf(y2, -1.1470745597729725e-11f, 2.0876756987868099e-9f);
    pc = fmaf(y2, pc, -2.7557319223985891e-7f);
    pc = fmaf(y2, pc, 2.4801587301587302e-5f);
    pc = fmaf(y2, pc, -1.3888888888888889e-3f);
    pc = fmaf(y2, pc, 4.1666666666666667e-2f);
    pc = fmaf(y2, pc, -0.5f);
    c = fmaf(y2, pc, 1.0f);
}

// e^{ikr}/r in FP32 from an FP32 r^2.  k r is reduced by pi (Cody-Waite, two-term split of
// pi: float(pi) and its remainder) to y in [-pi/2, pi/2], so that e^{ikr} = (-1)^n e^{iy}:
// the sign goes into 1/r as one bit.
HFMM_HD inline void radian_weight(float r2, float k, float& wr, float& wi) {
    const float rinv = rsq(r2);
    const float x = k * (r2 * rinv);
    const float kn = rintf(x * 0.318309886183790672f);
    float y = fmaf(-kn, 3.14159274101257324219f, x);
    y = fmaf(-kn, -8.74227800037248e-8f, y);
    float s, c;
    sincos_halfpi(y, s, c);
    const float rs = bitsf(fbits(rinv) ^ ((uint32_t)((int)kn & 1) << 31));
    wr = c * rs;
    wi = s * rs;
}

// e^{ikr}/r in FP32 with the phase k r accurate to FP64 rounding, from an FP64 r^2: r is
// the FP32 estimate r2 rsq(r2) refined by one Newton step in FP64, k r is reduced by pi
// (two-term FP64 split of pi) to y in [-pi/2, pi/2].  Also returns 1/r (positive) and k r
// (FP32) for the field weights.
HFMM_HD inline void radian_weight_phase64(double r2, double k, float& wr, float& wi, float& rinv, float& kr) {
    const float r2f = (float)r2;
    rinv = rsq(r2f);
    const double r0 = (double)(r2f * rinv);
    const double r = fma(0.5 * (double)rinv, fma(-r0, r0, r2), r0);
    const double ph = k * r;
    const double kn = rint(ph * 0.31830988618379067154);
    double y = fma(-kn, 3.1415926535897931160, ph);
    y = fma(-kn, 1.2246467991473532072e-16, y);
    float s, c;
    sincos_halfpi((float)y, s, c);
    const float rs = bitsf(fbits(rinv) ^ ((uint32_t)((int)kn & 1) << 31));
    wr = c * rs;
    wi = s * rs;
    kr = (float)ph;
}

}  // namespace nearfield
}  // namespace hfmm
