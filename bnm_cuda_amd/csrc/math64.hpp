// math64.hpp -- FP64 exponential, logarithm and reciprocal of the row-blocked and
// multi-workgroup integration kernels, and the row-blocked kernel's
// Balloon-Windkessel step made of them.
#pragma once
#include <hip/hip_runtime.h>

#include "model.hpp"

namespace bnm {

// FP64 reciprocal: the hardware estimate and one step of third order
// (y (1 + e + e^2), e = 1 - d y), about 1 ulp.
__device__ __forceinline__ double rcp_f64(double d) {
    const double y = __builtin_amdgcn_rcp(d);
    const double e = fma(-d, y, 1.0);
    return fma(y, fma(e, e, e), y);
}

// FP64 e^y by the reduction of Cody and Waite (1980), y = n ln 2 + f with ln 2 in two
// parts and |f| <= ln 2 / 2: e^y = 2^n (1 + m), m = e^f - 1 = f + f^2 Q(f), Q the
// degree-9 interpolant of (e^f - 1 - f) / f^2 at Chebyshev nodes (|error| of
// e^f <= 1.3e-17).  exp_parts returns m and n.
__device__ __forceinline__ double exp_parts(double y, double& n) {
    n = __builtin_rint(y * kLog2e);
    const double f = fma(-n, 0x1.a39ef35793c76p-33, fma(-n, 0x1.62e42fee00000p-1, y));
    const double f2 = f * f, f4 = f2 * f2;
    const double q01 = fma(f, 0x1.5555555555556p-3, 0x1.0000000000001p-1);
    const double q23 = fma(f, 0x1.11111111109b4p-7, 0x1.5555555553d67p-5);
    const double q45 = fma(f, 0x1.a01a01a7c327ap-13, 0x1.6c16c1788a49bp-10);
    const double q67 = fma(f, 0x1.71de0db21e27fp-19, 0x1.a019b9133a48ap-16);
    const double q89 = fma(f, 0x1.af38a0d2d9620p-26, 0x1.28917e2c43a66p-22);
    const double q = fma(f4, fma(f4, q89, fma(f2, q67, q45)), fma(f2, q23, q01));
    return fma(f2, q, f);
}

// 1 - e^y, within 3 ulp for every y, also next to y = 0, where the difference of a
// rounded e^y from 1 has few digits left: (1 - 2^n) - 2^n m, whose first term is exact
// for n >= -53 and zero for n = 0.  y is cut off at 700, where 1 / (1 - e^y) and
// everything made of it is zero next to any value of the model.  Not for -infinity
// (NaN) and NaN (cut off too): see Pool<double>::rate().
__device__ __forceinline__ double one_minus_exp_f64(double y) {
    double n;
    const double m = exp_parts(fmin(y, 700.0), n);
    const double t = __builtin_ldexp(1.0, (int)n);
    return fma(-t, m, 1.0 - t);
}

// e^y, about 1 ulp; y is cut off as above, and is not -infinity or NaN.
__device__ __forceinline__ double exp_f64(double y) {
    double n;
    const double m = exp_parts(fmin(y, 700.0), n);
    return __builtin_ldexp(1.0 + m, (int)n);
}

// ln v, FP64, as hi + lo (v > 0 and finite): v = 2^e m with m in [sqrt 1/2, sqrt 2),
// ln m = 2 s + s^3 W(s^2), s = (m - 1) / (m + 1), W the degree-6 interpolant at
// Chebyshev nodes (relative error <= 5e-18 of the series).  s is rounded, and so is the
// m + 1 that it is a quotient by: sl is what s is short of.  hi is the rounded
// logarithm, lo what that leaves.
__device__ __forceinline__ double log_parts(double v, double& lo) {
    double m = __builtin_amdgcn_frexp_mant(v);
    int e = __builtin_amdgcn_frexp_exp(v);
    const bool low = m < 0.70710678118654752;
    m = low ? m + m : m;
    e = low ? e - 1 : e;
    const double d = m - 1.0, b = m + 1.0;
    const double rb = rcp_f64(b), s = d * rb, z = s * s;
    const double sl = fma(-s, m - (b - 1.0), fma(-s, b, d)) * rb;   // (b + (m - (b - 1)) = m + 1)
    double w = 0x1.2b5f68a50d903p-3;
    w = fma(w, z, 0x1.39fdcceb4bb45p-3);
    w = fma(w, z, 0x1.7462b91b8df65p-3);
    w = fma(w, z, 0x1.c71c62d5e53e0p-3);
    w = fma(w, z, 0x1.2492492dfd86cp-2);
    w = fma(w, z, 0x1.9999999995273p-2);
    w = fma(w, z, 0x1.5555555555558p-1);
    const double n = (double)e, big = n * 0x1.62e42fee00000p-1;   // (exact, and above 2 s or zero)
    const double h = big + (s + s);
    const double l = ((big - h) + (s + s)) + fma(n, 0x1.a39ef35793c76p-33, fma(s * z, w, sl + sl));
    const double hi = h + l;
    lo = l - (hi - h);
    return hi;
}

// v^p for hi + lo = ln v; NaN unless v is positive and finite (logarithm and
// exponential have finite values for zero and negative v, and a run that gets there is
// to end in NaN, as with pow).
__device__ __forceinline__ double pow_f64(double hi, double lo, double p, double v) {
    const double y = p * hi, e = exp_f64(y);
    const double r = fma(e, fma(p, lo, fma(p, hi, -y)), e);
    return v > 0.0 && v < __builtin_inf() ? r : __builtin_nan("");
}

// Balloon-Windkessel step in six parts, so that the row-blocked kernel can run
// it between the LDS reads of the next millisecond's substeps.  From rest (x =
// 0, f = nu = q = 1) a step with S_E = 0 changes nothing.
template <class T> struct BWParts;

// FP32: the operations of BW<float>, selects in place of its branches
template <> struct BWParts<float> : BW<float> {
    float f1, u, q1, lg, E, un, En, em;
    double fmn;
    static __device__ __forceinline__ float expm1s(float z) {
        float p = 1.0f / 362880.0f;
        p = fmaf(p, z, 1.0f / 40320.0f);
        p = fmaf(p, z, 1.0f / 5040.0f);
        p = fmaf(p, z, 1.0f / 720.0f);
        p = fmaf(p, z, 1.0f / 120.0f);
        p = fmaf(p, z, 1.0f / 24.0f);
        p = fmaf(p, z, 1.0f / 6.0f);
        p = fmaf(p, z, 0.5f);
        p = fmaf(p, z, 1.0f);
        const float far = __builtin_amdgcn_exp2f(z * (float)kLog2e) - 1.0f;
        return fabsf(z) > 0.5f ? far : p * z;
    }
    template <int K>
    __device__ __forceinline__ void part(float SE) {
        constexpr float mdt = (float)C64::model_dt;
        constexpr float mdt_itau = (float)(C64::model_dt * C64::itau);
        constexpr float kap = (float)C64::kappa, yy = (float)C64::y;
        constexpr float ia = (float)C64::ialpha;
        constexpr float c1 = (float)(C64::oneminrho / C64::rho);
        constexpr float c2 = (float)(-kLog2OneMinRho / kLog2e);
        if constexpr (K == 0) {
            const float xf = (float)x;
            f1 = (float)fm;
            u = (float)um;
            q1 = (float)qm;
            x += (double)(mdt * (SE - kap * xf - yy * f1));
            fmn = fm + (double)(mdt * (float)x);
        } else if constexpr (K == 1) {
            const float s = u * __builtin_amdgcn_rcpf(2.0f + u);
            const float s2 = s * s;
            float p = 1.0f / 11.0f;
            p = fmaf(p, s2, 1.0f / 9.0f);
            p = fmaf(p, s2, 1.0f / 7.0f);
            p = fmaf(p, s2, 1.0f / 5.0f);
            p = fmaf(p, s2, 1.0f / 3.0f);
            p = fmaf(p, s2, 1.0f);
            const float far = __builtin_amdgcn_logf(1.0f + u) * (float)(1.0 / kLog2e);
            lg = fabsf(s) > 0.15f ? far : 2.0f * s * p;
        } else if constexpr (K == 2) {
            E = expm1s(ia * lg);
        } else if constexpr (K == 3) {
            const float ru = __builtin_amdgcn_rcpf(1.0f + u);
            const float dnu = mdt_itau * (f1 - E);
            um += (double)dnu;
            un = (float)um;
            En = fmaf(ia * (1.0f + E) * ru, dnu, E);
        } else if constexpr (K == 4) {
            em = expm1s(c2 * f1 * __builtin_amdgcn_rcpf(1.0f + f1));
        } else {
            const float t1 = f1 - (1.0f + f1) * c1 * em;
            const float t2 = (En + q1 + En * q1 - un) * __builtin_amdgcn_rcpf(1.0f + un);
            qm += (double)(mdt_itau * (t1 - t2));
            fm = fmn;
        }
    }
};

// FP64: the step of BW<double> with products by reciprocals, exp_f64 and
// log_parts, and nu^(1/alpha) kept from one step for the next (a step's new nu
// is the next one's old nu)
template <> struct BWParts<double> {
    double x, f, nu, q, pn, fn, lg, lgl, E, rn;
    __device__ __forceinline__ void reset() { x = 0.0; f = nu = q = pn = 1.0; }
    template <int K>
    __device__ __forceinline__ void part(double SE) {
        constexpr double kLnOneMinRho = -0x1.a97ce16b316f4p-2;   // ln(1 - rho), 1 - rho rounded to FP64
        if constexpr (K == 0) {
            x = fma(C64::model_dt, fma(-C64::y, f - 1.0, fma(-C64::kappa, x, SE)), x);
            fn = fma(C64::model_dt, x, f);
            nu = fma(C64::model_dt * C64::itau, f - pn, nu);
        } else if constexpr (K == 1) {
            lg = log_parts(nu, lgl);
        } else if constexpr (K == 2) {
            pn = pow_f64(lg, lgl, C64::ialpha, nu);
        } else if constexpr (K == 3) {
            E = kLnOneMinRho * rcp_f64(f);
            rn = rcp_f64(nu);
        } else if constexpr (K == 4) {
            E = 1.0 - exp_f64(E);
        } else {
            q = fma(C64::model_dt * C64::itau, fma(f * E, 1.0 / C64::rho, -(pn * q * rn)), q);
            f = fn;
        }
    }
    __device__ __forceinline__ double bold(double k1, double k2, double k3) const {
        return C64::V0 * (k1 * (1 - q) + k2 * (1 - q / nu) + k3 * (1 - nu));
    }
};

}  // namespace bnm
