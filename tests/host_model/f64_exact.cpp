// The FP64 functions of math64.hpp, and whole runs of Pool<double> and
// BWParts<double>, against 128-bit arithmetic on the host, beside runs of
// Node<double> and BW<double> (the reference's order of operations, exp and pow of
// the host's libm) on the same inputs.
//
// "f64_exact functions": largest error in ulp of each function over its ranges.
// "f64_exact edges": number of cases in which infinite, undefined or far couplings
// give another S or r than Node<double>, or a Balloon-Windkessel state whose nu is
// zero, negative, infinite or undefined gives finite BOLD.
// "f64_exact runs T sims": N = 6 nodes coupled by a random SC, T ms, `sims` parameter
// sets; prints the rms errors of S_E (every ms) and of BOLD (every 100 ms) of both,
// over all sets, each set's errors divided by its largest value.
#include <quadmath.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include <hip/hip_runtime.h>

// the lane exchange hands on the partner's value, set before each use
static int partner_half[2], partner_at;
inline int __builtin_amdgcn_update_dpp(int, int, int, int, int, bool) { return partner_half[partner_at++ & 1]; }
// the hardware's reciprocal estimate, good to 2^-24
inline double __builtin_amdgcn_rcp(double d) {
    int e;
    const double m = std::frexp(1.0 / d, &e);
    return std::ldexp(std::rint(std::ldexp(m, 24)), e - 24);
}
inline double __builtin_amdgcn_frexp_mant(double v) { int e; return std::frexp(v, &e); }
inline int __builtin_amdgcn_frexp_exp(double v) { int e; std::frexp(v, &e); return e; }
template <class A, class B> static A bits(B b) { A a; std::memcpy(&a, &b, sizeof a); return a; }
inline long long __double_as_longlong(double d) { return bits<long long>(d); }
inline double __longlong_as_double(long long u) { return bits<double>(u); }
inline int __float_as_int(float f) { return bits<int>(f); }
inline float __int_as_float(int u) { return bits<float>(u); }

#include "../../bnm_cuda_amd/csrc/pool.hpp"

using namespace bnm;
typedef __float128 Q;

static void partner(double S) {
    const long long u = bits<long long>(S);
    partner_half[0] = (int)u;
    partner_half[1] = (int)(u >> 32);
    partner_at = 0;
}

template <class F, class E>
static void ulps(const char* name, double lo, double hi, bool log_x, F f, E exact) {
    std::mt19937_64 rng(3);
    std::uniform_real_distribution<double> U(lo, hi);
    double worst = 0;
    for (int i = 0; i < 300000; ++i) {
        double x = U(rng);
        if (log_x) x = (i & 1 ? -1 : 1) * std::exp(x);
        const Q ref = exact(x);
        int e;
        std::frexp((double)ref, &e);
        worst = std::max(worst, std::fabs((double)(((Q)f(x) - ref) / (Q)std::ldexp(1.0, e - 53))));
    }
    std::printf("%s %.4f\n", name, worst);
}

static double log64(double v) { double lo; const double hi = log_parts(v, lo); return hi + lo; }
static double pow64(double v) {
    double lo;
    const double hi = log_parts(v, lo);
    return pow_f64(hi, lo, C64::ialpha, v);
}

static void functions() {
    ulps("exp", -40, 40, false, [](double x) { return exp_f64(x); }, [](double x) { return expq(x); });
    ulps("log", 0.3, 3, false, log64, [](double x) { return logq(x); });
    ulps("log_near_1", 0.9, 1.1, false, log64, [](double x) { return logq(x); });
    ulps("pow", 0.5, 2, false, pow64, [](double x) { return powq(x, C64::ialpha); });
    auto d = [](double x) { return one_minus_exp_f64(x); };
    auto dq = [](double x) { return -expm1q(x); };
    ulps("one_minus_exp", -40, 40, false, d, dq);
    ulps("one_minus_exp_small", -30, 0, true, d, dq);
}

// NaN for NaN, infinity for infinity, otherwise to rel: 1e-13, what cancellation in x
// leaves, a difference of two values about 125 (one rounding 1.4e-14 each, |x| above 1
// here)
static int differ(const char* what, double x, double got, double want, double rel) {
    const bool same = want != want ? got != got : want == got || std::fabs(got - want) <= rel * std::fabs(want);
    if (!same) std::fprintf(stderr, "%s(%g) = %g, not %g\n", what, x, got, want);
    return !same;
}

static void edges() {
    const double inf = INFINITY, nan = NAN;
    int bad = 0;
    for (double v : std::vector<double>{0.0, -1e-9, -0.5, -1.0, -3e7, inf, nan}) {
        BWParts<double> b;
        b.reset();
        for (int step = 0; step < 3; ++step) {
            b.nu = step ? b.nu : v;
            b.part<0>(0.1); b.nu = step ? b.nu : v;
            b.part<1>(0.1); b.part<2>(0.1); b.part<3>(0.1); b.part<4>(0.1); b.part<5>(0.1);
        }
        const double B = b.bold(C64::k1, C64::k2, C64::k3);
        if (B == B) { std::fprintf(stderr, "BOLD for nu = %g: %g\n", v, B); ++bad; }
    }
    for (double v : std::vector<double>{0.0, 1.0, 1e4, 1e9, 1e30, inf, -1e3, -1e9, -inf, nan}) {
        double SE = 0.001, SI = 0.001, IE, II, rE, rI;
        Node<double>::step(v, 1.0, 0.2, 0.2, 1.0, 0.125, 0.125, SE, SI, IE, II, rE, rI);
        Pool<double> e;
        e.init(0, 1.0, 0.2, 0.2, 1.0);
        partner(0.001);
        e.before(0.125f);
        e.after(v, true);
        // (for a far negative x the rate is zero beside anything: below 1e-200)
        bad += differ("S_E", v, e.S, SE, 1e-13) +
               differ("r_E", v, std::fabs(e.rate()) < 1e-200 ? 0.0 : e.rate(), std::fabs(rE) < 1e-200 ? 0.0 : rE, 1e-13);
    }
    std::printf("edges %d\n", bad);
}

struct Exact {
    Q SE = 0.001, SI = 0.001, x = 0, f = 1, nu = 1, q = 1;
    void substep(Q c, double G, double wEE, double wEI, double wIE, float xiE, float xiI) {
        const Q I = (Q)C64::wE_I0 + (Q)wEE * SE + c * G * (Q)C64::J_NMDA - (Q)wIE * SI;
        const Q J = (Q)C64::wI_I0 + (Q)wEI * SE - SI;
        const Q u = (Q)C64::a_E * I - C64::b_E, v = (Q)C64::a_I * J - C64::b_I;
        const Q r = u / (1 - expq(-(Q)C64::d_E * u)), s = v / (1 - expq(-(Q)C64::d_I * v));
        const Q nz = (Q)C64::sigma * (Q)C64::sqrt_dt;
        SE += xiE * nz + (Q)C64::dt * ((1 - SE) * (Q)C64::gamma_E * r - SE / C64::tau_E);
        SI += xiI * nz + (Q)C64::dt * ((Q)C64::gamma_I * s - SI / C64::tau_I);
        SE = SE < 0 ? 0 : SE > 1 ? 1 : SE;
        SI = SI < 0 ? 0 : SI > 1 ? 1 : SI;
    }
    void bw() {
        x += (Q)C64::model_dt * (SE - (Q)C64::kappa * x - (Q)C64::y * (f - 1));
        const Q fn = f + (Q)C64::model_dt * x, h = (Q)C64::model_dt * (Q)C64::itau;
        nu += h * (f - powq(nu, C64::ialpha));
        q += h * (f * (1 - powq(C64::oneminrho, 1 / f)) / C64::rho - powq(nu, C64::ialpha) * q / nu);
        f = fn;
    }
    Q bold() const { return (Q)C64::V0 * (C64::k1 * (1 - q) + C64::k2 * (1 - q / nu) + C64::k3 * (1 - nu)); }
};

static void runs(int T, int sims) {
    const int N = 6;
    double S2[2] = {0, 0}, B2[2] = {0, 0};
    for (int sim = 0; sim < sims; ++sim) {
        std::mt19937 rng(sim);
        std::uniform_real_distribution<double> U(0, 1);
        std::normal_distribution<float> Z(0, 1);
        std::vector<double> SC(N * N, 0.0), wEE(N), wEI(N), wIE(N);
        double sum = 0;
        for (int i = 0; i < N; ++i)
            for (int j = 0; j < i; ++j) sum += 2 * (SC[i * N + j] = SC[j * N + i] = U(rng) < 0.6 ? U(rng) : 0.0);
        for (double& v : SC) v *= N / std::max(sum, 1.0);
        const double G = 0.5 + 2.5 * U(rng);
        for (int j = 0; j < N; ++j) {
            wEE[j] = 0.05 + 0.4 * U(rng);
            wEI[j] = 0.05 + 0.4 * U(rng);
            wIE[j] = 0.8 + 1.5 * U(rng);
        }
        std::vector<double> SE(N, 0.001), SI(N, 0.001), Sp(N), IE(N), II(N), rE(N), rI(N), Pe(N), Pi(N);
        std::vector<BW<double>> bw(N);
        std::vector<Pool<double>> e(N), i(N);
        std::vector<BWParts<double>> parts(N);
        std::vector<Exact> x(N);
        std::vector<Q> Qp(N);
        for (int j = 0; j < N; ++j) {
            e[j].init(0, G, wEE[j], wEI[j], wIE[j]);
            i[j].init(1, G, wEE[j], wEI[j], wIE[j]);
            parts[j].reset();
        }
        double s2[2] = {0, 0}, b2[2] = {0, 0}, smax = 0, bmax = 0;
        long nb = 0;
        for (int ts = 0; ts <= T; ++ts) {
            for (int k = 0; k < 10; ++k) {
                Sp = SE;
                for (int j = 0; j < N; ++j) {
                    Pe[j] = e[j].S;
                    Pi[j] = i[j].S;
                    Qp[j] = x[j].SE;
                }
                for (int j = 0; j < N; ++j) {
                    const float xe = Z(rng), xi = Z(rng);
                    double c = 0, d = 0;
                    Q cq = 0;
                    for (int m = 0; m < N; ++m) {
                        c = std::fma(SC[j * N + m], Sp[m], c);
                        d = std::fma(SC[j * N + m], Pe[m], d);
                        cq += (Q)SC[j * N + m] * Qp[m];
                    }
                    Node<double>::step(c, G, wEE[j], wEI[j], wIE[j], xe, xi, SE[j], SI[j], IE[j], II[j], rE[j], rI[j]);
                    partner(Pi[j]);
                    e[j].before(xe);
                    partner(Pe[j]);
                    i[j].before(xi);
                    e[j].after(d, true);
                    i[j].after(d, true);
                    x[j].substep(cq, G, wEE[j], wEI[j], wIE[j], xe, xi);
                }
            }
            for (int j = 0; j < N; ++j) {
                BWParts<double>& p = parts[j];
                const double S = e[j].S;
                bw[j].step(SE[j]);
                p.part<0>(S); p.part<1>(S); p.part<2>(S); p.part<3>(S); p.part<4>(S); p.part<5>(S);
                x[j].bw();
                const double a = (double)(SE[j] - x[j].SE), b = (double)(S - x[j].SE);
                s2[0] += a * a;
                s2[1] += b * b;
                smax = std::max(smax, S);
                if (ts % 100) continue;
                const Q B = x[j].bold();
                const double u = (double)(bw[j].bold(C64::k1, C64::k2, C64::k3) - B);
                const double v = (double)(p.bold(C64::k1, C64::k2, C64::k3) - B);
                b2[0] += u * u;
                b2[1] += v * v;
                bmax = std::max(bmax, std::fabs((double)B));
                ++nb;
            }
        }
        for (int w = 0; w < 2; ++w) {
            S2[w] += s2[w] / (N * (T + 1.0)) / (smax * smax);
            B2[w] += b2[w] / nb / (bmax * bmax);
        }
    }
    std::printf("S_reference %.6e\nS_kernels %.6e\n", std::sqrt(S2[0] / sims), std::sqrt(S2[1] / sims));
    std::printf("BOLD_reference %.6e\nBOLD_kernels %.6e\n", std::sqrt(B2[0] / sims), std::sqrt(B2[1] / sims));
}

int main(int argc, char** argv) {
    if (argc == 2 && !std::strcmp(argv[1], "functions")) functions();
    else if (argc == 2 && !std::strcmp(argv[1], "edges")) edges();
    else if (argc == 4) runs(std::atoi(argv[2]), std::atoi(argv[3]));
    else return 2;
    return 0;
}
