// pool.hpp -- one pool's update per lane and the lane exchanges of the
// row-blocked and multi-workgroup integration kernels: the excitatory pool of a
// node in an even lane, its inhibitory pool in the odd lane next to it.
#pragma once
#include <hip/hip_runtime.h>

#include "math64.hpp"
#include "model.hpp"

namespace bnm {

namespace {

// DPP moves within a 16-lane row
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kMirror8 = 0x141, kMirror16 = 0x140;

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// LDS writes of this wave done, then the workgroup barrier (global loads in
// flight stay in flight)
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <class T> struct Pool;

// strict FP32 update of one pool in own / other form: k_S multiplies this
// lane's S, k_O the partner's
template <> struct Pool<float> {
    float k0h, k0l, kSh, kSl, kOh, kOl, ch, cl, GJ, aa, bb, ndlh, ndll, invd, d12, g, gl, gm, gml, it, itl;
    float S, Sl, r, I;
    float pre, prel, X0, A, Al, D;   // formed before the coupling arrives
    float u, t, Sp;
    double wIE;
    __device__ __forceinline__ void init(int pop, double G, double wEE, double wEI, double w) {
        const bool e = pop == 0;
        const double a = e ? C64::a_E : C64::a_I, d = e ? C64::d_E : C64::d_I;
        const double g64 = C64::dt * (e ? C64::gamma_E : C64::gamma_I);
        const double it64 = C64::dt / (e ? C64::tau_E : C64::tau_I);
        NodeStrict::split(e ? C64::wE_I0 : C64::wI_I0, k0h, k0l);
        NodeStrict::split(e ? wEE : -1.0, kSh, kSl);
        NodeStrict::split(e ? -w : wEI, kOh, kOl);
        NodeStrict::split(e ? a * (G * C64::J_NMDA) : 0.0, ch, cl);
        GJ = e ? (float)(G * C64::J_NMDA) : 0.0f;
        aa = (float)a;
        bb = (float)(e ? C64::b_E : C64::b_I);
        NodeStrict::split(-d * kLog2e, ndlh, ndll);
        invd = (float)(1.0 / d);
        d12 = (float)(d / 12.0);
        NodeStrict::split(g64, g, gl);
        gm = e ? g : 0.0f;
        gml = e ? gl : 0.0f;
        NodeStrict::split(it64, it, itl);
        wIE = w;
        r = I = 0.0f;
        reset();
    }
    __device__ __forceinline__ void reset() { S = 0.001f; Sl = NodeStrict::kS0l; }
    __device__ __forceinline__ void set_wIE(bool e) { if (e) NodeStrict::split(-wIE, kOh, kOl); }
    __device__ __forceinline__ double value() const { return (double)S + (double)Sl; }
    __device__ __forceinline__ double rate() const { return (double)r; }
    __device__ __forceinline__ void before(float xi) {
        constexpr double nzs64 = C64::sigma * C64::sqrt_dt;
        constexpr float nzs = (float)nzs64, nzsl = (float)(nzs64 - (double)nzs);
        const float So = dpp<kXor1>(S);
        pre = fmaf(kOh, So, fmaf(kSh, S, k0h));
        prel = fmaf(kOl, So, fmaf(kSl, S, k0l));
        X0 = fmaf(aa, prel, fmaf(aa, pre, -bb));
        A = fmaf(-gm, S, g);
        Al = fmaf(-gml, S, gl);
        D = fmaf(xi, nzsl, fmaf(-itl, S, fmaf(-it, S, xi * nzs))) + Sl;
    }
    __device__ __forceinline__ void after(float c, bool last) {
        if (last) I = fmaf(GJ, c, pre) + prel;
        const float x = fmaf(ch, c, fmaf(cl, c, X0));
        const float y = fmaf(ndlh, x, ndll * x);
        const float direct = x * __builtin_amdgcn_rcpf(1.0f - __builtin_amdgcn_exp2f(y));
        const float series = invd + x * (0.5f + d12 * x);
        r = fabsf(x) < 0.1f ? series : direct;
        u = fmaf(r, A, fmaf(r, Al, D));
        Sp = S;
        t = S + u;
        S = __builtin_amdgcn_fmed3f(t, 0.0f, 1.0f);
    }
    // the low part of S, once S is on its way to the other waves
    __device__ __forceinline__ void settle() { Sl = S == t ? u - (t - Sp) : 0.0f; }
};

// FP64, contracted, as exact as the reference's order of operations or more so: the
// increment of S is formed first, so that S takes one rounding of its own magnitude a
// substep (three, as a chain of fused operations on S, doubled its error), and 1 - e^y
// keeps its digits where x is small.
template <> struct Pool<double> {
    double k0, kS, kO, ac, GJ, aa, bb, nd, g, gm, it;
    double S, r, I;
    double pre, X0, A, D;
    double wIE;
    __device__ __forceinline__ void init(int pop, double G, double wEE, double wEI, double w) {
        const bool e = pop == 0;
        k0 = e ? C64::wE_I0 : C64::wI_I0;
        kS = e ? wEE : -1.0;
        kO = e ? -w : wEI;
        aa = e ? C64::a_E : C64::a_I;
        bb = e ? C64::b_E : C64::b_I;
        GJ = e ? G * C64::J_NMDA : 0.0;
        ac = aa * GJ;
        nd = e ? -C64::d_E : -C64::d_I;
        g = C64::dt * (e ? C64::gamma_E : C64::gamma_I);
        gm = e ? g : 0.0;
        it = C64::dt / (e ? C64::tau_E : C64::tau_I);
        wIE = w;
        r = I = 0.0;
        reset();
    }
    __device__ __forceinline__ void reset() { S = 0.001; }
    __device__ __forceinline__ void set_wIE(bool e) { if (e) kO = -wIE; }
    __device__ __forceinline__ double value() const { return S; }
    // r of the last substep, also for an infinite I, where after() leaves NaN (S is 1
    // either way)
    __device__ __forceinline__ double rate() const {
        return fabs(I) < 1e300 ? r : I > 0.0 ? __builtin_inf() : __builtin_nan("");
    }
    __device__ __forceinline__ void before(float xi) {
        constexpr double nzs = C64::sigma * C64::sqrt_dt;
        const double So = dpp<kXor1>(S);
        pre = fma(kO, So, fma(kS, S, k0));
        X0 = fma(aa, pre, -bb);
        A = fma(-gm, S, g);
        D = fma(-it, S, (double)xi * nzs);
    }
    __device__ __forceinline__ void after(double c, bool last) {
        if (last) I = fma(GJ, c, pre);
        const double x = fma(ac, c, X0);
        r = x * rcp_f64(one_minus_exp_f64(nd * x));
        S = fmax(0.0, fmin(S + fma(r, A, D), 1.0));
    }
    __device__ __forceinline__ void settle() {}
};

}  // namespace

}  // namespace bnm
