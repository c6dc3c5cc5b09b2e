// sim_block.hip -- integration kernel with the coupling product blocked over
// rows, one simulation per workgroup, all of SC in VGPRs.
//
// Wave w holds nodes 32 w .. 32 w + 31, two lanes a node: lane l steps pool
// l & 1 (0 excitatory, 1 inhibitory) of node 32 w + l / 2, so that its draw is
// at 2 j + pool and a wave's noise is 256 contiguous bytes.  The product SC S_E
// is split over groups of Q = 2 R lanes: each lane of a group multiplies R rows
// (the group's R nodes) with its own k-slice of KC = ceil(N / Q) values.  The
// sums then go to the lanes that need them in log2 Q DPP adds: at each step a
// lane keeps the rows of its own half of the group and takes from its mirror
// image the sums that it has made for them; its accumulators are ordered so
// (block_row) that no select is needed, and the last step leaves the node's sum
// in both its lanes.
//
// What bounds it: one substep is a serial chain, one wave per SIMD (N <= 128).
// At N = 100 in FP32 of 673 cycles 207 are the FMAs (52 per lane, four cycles
// each), about 270 the way of S through LDS (write, barrier, read) and the sum
// over lanes, 115 + 45 the update after and before the coupling, 35 the BW
// step.  Against one row per lane (k_sim_ei: 907 cycles) a lane reads 13
// values from LDS where it read 52, and the reads no longer compete with the
// FMAs for the register file.  R = 4 against 2 and 8: 673, 691, 683 cycles
// (FP64 775, 852, 828).  What does not wait for the coupling is formed before
// the barrier, the BW step runs in parts between the LDS reads of the next
// millisecond's substeps, and each substep's noise is loaded a millisecond
// ahead into the register that its last draw has left.
//
// FP32 is the strict update (hi / lo coefficients as NodeStrict) in own /
// partner form.  FP64 uses fused multiply-adds, the functions of math64.hpp and
// reciprocals of the constants in place of the reference's order of operations
// (k_sim_ei64, in that order: 1758 cycles).
#include <algorithm>

#include "kernels.hpp"
#include "model.hpp"
#include "pool.hpp"

namespace bnm {

namespace {

// Node of the wave's group whose product with slice q is a lane's r-th
// accumulator (see k_sim_block)
__device__ __forceinline__ int block_row(int q, int r) {
    if (r & 4) q = 15 - q;
    if (r & 2) q = (q & 8) | (7 - (q & 7));
    return (q >> 1) ^ (r & 1);
}

}  // namespace

template <class T, int R, int KC>
__device__ __forceinline__ void block_run(const T* __restrict__ SC, const SimArgs& a, int SS) {
    constexpr int Q = 2 * R;                       // lanes of a group, k-slices
    constexpr int VW = 16 / sizeof(T);
    typedef T vec __attribute__((ext_vector_type(VW)));
    const int sim = blockIdx.x;
    const int N = a.N;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q = lane & (Q - 1), pop = lane & 1;
    const int j = wave * 32 + (lane >> 1);
    const int j0 = j - (q >> 1);                    // the group's first node
    const bool comp = j < N;
    const bool writer = comp && pop == 0;
    const int jc = comp ? j : N - 1;                // lanes past the last node run node N - 1's update
    const int ldS = Q * SS;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* Sb = reinterpret_cast<T*>(smem_raw);         // [2][ldS], then 64 slots nobody reads
    T sc[R][KC];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = j0 + block_row(q, r);
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            const int k = q * KC + i;
            sc[r][i] = (row < N && k < N) ? SC[(size_t)row * N + k] : T(0);
        }
    }
    for (int i = threadIdx.x; i < 2 * ldS; i += blockDim.x) {
        const int slot = i % ldS, qq = slot % SS, k = (slot / SS) * KC + qq;
        Sb[i] = (qq < KC && k < N) ? T(0.001) : T(0);
    }
    const T* Sr = Sb + q * SS;
    // where the lane's S goes: the node's slot, or a slot that nobody reads
    const int pos0 = writer ? (j / KC) * SS + j % KC : 2 * ldS + lane;
    const int pos1 = writer ? ldS + pos0 : pos0;

    const size_t o = (size_t)sim * N + jc;
    Pool<T> p;
    p.init(pop, a.G[sim], a.wEE[o], a.wEI[o], a.wIE_in[o]);
    double delta = a.init_delta;
    BWParts<T> bw;
    bw.reset();
    T bwS = 0;                                      // S_E of the millisecond that the BW step is behind by
    int bold_vol = -1;                              // the volume that millisecond is, if it is one
    double mI = 0, ext[3] = {0, 0, 0};
    int ts = 0, vol = 0, trial = 0, next_vol = 0;
    bool adjusting = a.adjust_fic != 0, failed = false;
    const unsigned dur = (unsigned)(a.i_end - a.i_start + 1);
    const int P = (int)a.noise_period;
    // noise: nz[s] holds substep s's draw until its update, then the next
    // millisecond's is loaded in its place
    const unsigned noff = (unsigned)(2 * jc + pop) * (unsigned)sizeof(float);
    auto draw = [&](int ms, int s) {
        const float* row = a.noise + ((size_t)ms * 10 + s) * 2 * N;
        return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(row) + noff);
    };
    auto store_bold = [&](int v) {
        if (writer)
            reinterpret_cast<T*>(a.bold)[((size_t)sim * a.output_ts + v) * N + j] =
                (T)bw.bold(a.bw_k1, a.bw_k2, a.bw_k3);
    };
    float nz[10];
    int ms1 = P > 1 ? 1 : 0;                        // the next millisecond's place in the noise
#pragma unroll
    for (int s = 0; s < 10; ++s) nz[s] = draw(0, s);
    p.before(nz[0]);
    nz[0] = draw(ms1, 0);
    __syncthreads();
    while (ts <= a.time_steps) {
        const int ms2 = ms1 + 1 == P ? 0 : ms1 + 1;
#pragma unroll
        for (int s = 0; s < 10; ++s) {
            const T* Sx = Sr + (s & 1) * ldS;
            T v[KC];
#pragma unroll
            for (int i = 0; i + VW <= KC; i += VW) {
                const vec t = *reinterpret_cast<const vec*>(Sx + i);
#pragma unroll
                for (int w = 0; w < VW; ++w) v[i + w] = t[w];
            }
#pragma unroll
            for (int i = KC / VW * VW; i < KC; ++i) v[i] = Sx[i];
            // a part of the last millisecond's BW step while the reads are under way
            if (s == 1) bw.template part<0>(bwS);
            if (s == 2) bw.template part<1>(bwS);
            if (s == 3) bw.template part<2>(bwS);
            if (s == 4) bw.template part<3>(bwS);
            if (s == 5) bw.template part<4>(bwS);
            if (s == 6) bw.template part<5>(bwS);
            T acc[R];
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] = sc[r][0] * v[0];
#pragma unroll
            for (int i = 1; i < KC; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r) acc[r] = fma(sc[r][i], v[i], acc[r]);
            if constexpr (R == 8)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r] += dpp<kMirror16>(acc[r + 4]);
            if constexpr (R >= 4)
#pragma unroll
                for (int r = 0; r < 2; ++r) acc[r] += dpp<kMirror8>(acc[r + 2]);
            T c = acc[0];
            if constexpr (R >= 2) c += dpp<kXor2>(acc[1]);
            c += dpp<kXor1>(c);
            p.after(c, s == 9);
            Sb[(s & 1) ? pos0 : pos1] = p.S;
            p.settle();
            if (s < 9) {
                p.before(nz[s + 1]);
                nz[s + 1] = draw(ms1, s + 1);
            } else {
                p.before(nz[0]);
                nz[0] = draw(ms2, 0);
            }
            lds_barrier();
        }
        ms1 = ms2;
        if (bold_vol >= 0) store_bold(bold_vol);
        bold_vol = -1;
        bwS = p.S;
        if (ts == next_vol) {
            next_vol += a.bold_tr;
            bold_vol = vol;
            if (vol >= a.n_vols_remove) {
                ext[0] += p.value();
                ext[1] += (double)p.I;
                ext[2] += p.rate();
            }
            ++vol;
        }
        ++ts;
        if (adjusting) {
            if (ts >= a.i_start && ts <= a.i_end) mI += (double)p.I;
            if (ts == a.i_end) {
                // the excitatory lane decides; the inhibitory pool has no wIE
                const bool out = writer && fic_decide<double>(mI, dur, trial, a.max_fic_trials, p.wIE, delta);
                p.set_wIE(pop == 0);
                if (__syncthreads_or(out)) {
                    if (trial < a.max_fic_trials) {
                        p.reset();
                        bw.reset();
                        bwS = 0;
                        bold_vol = -1;
                        mI = 0;
                        ext[0] = ext[1] = ext[2] = 0;
                        Sb[pos0] = p.S;
                        ts = 0; vol = 0; next_vol = 0; ++trial;
                        ms1 = P > 1 ? 1 : 0;
#pragma unroll
                        for (int s = 0; s < 10; ++s) nz[s] = draw(0, s);
                        p.before(nz[0]);
                        nz[0] = draw(ms1, 0);
                        __syncthreads();
                    } else {
                        failed = true; adjusting = false;
                    }
                } else {
                    adjusting = false;
                }
            }
        }
    }
    bw.template part<0>(bwS);
    bw.template part<1>(bwS);
    bw.template part<2>(bwS);
    bw.template part<3>(bwS);
    bw.template part<4>(bwS);
    bw.template part<5>(bwS);
    if (bold_vol >= 0) store_bold(bold_vol);
    if (comp) {
        if (pop == 0) a.wIE_out[o] = p.wIE;
        const int n = vol - a.n_vols_remove;
        for (int i = 0; i < 3; ++i) a.ext[((size_t)sim * 6 + 3 * pop + i) * N + j] = n > 0 ? ext[i] / n : 0.0;
    }
    if (threadIdx.x == 0) {
        a.fic_failed[sim] = failed ? 1 : 0;
        a.fic_trials[sim] = trial;
    }
}

template <class T, int R, int KC, int MAXT, int WAVES>
__global__ __launch_bounds__(MAXT, WAVES) void k_sim_block(const T* __restrict__ SC, SimArgs a, int SS) {
    block_run<T, R, KC>(SC, a, SS);
}
// no more than MOST waves a SIMD
template <class T, int R, int KC, int MAXT, int MOST>
__global__ __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(MOST, MOST))) void k_sim_block_most(
    const T* __restrict__ SC, SimArgs a, int SS) {
    block_run<T, R, KC>(SC, a, SS);
}

// KC: slice lengths that the kernel is built for; R = 4 rows a lane.  FP64 takes
// up to 128 nodes (16 values x 4 rows = 128 VGPRs); FP32 up to 256, with two
// waves a SIMD from 129 on.
static const int kBlockKC[] = {4, 6, 8, 10, 13, 16, 20, 25, 28, 32};

BlockShape block_shape(int N, size_t elem) {
    BlockShape s{};
    const int per = (N + 7) / 8;
    for (int kc : kBlockKC)
        if (kc >= per) { s.KC = kc; break; }
    // slices start 16 bytes x an odd number apart: the eight slices that a wave
    // reads at once lie in distinct banks
    const int vw = 16 / (int)elem;
    s.SS = (s.KC + vw - 1) / vw * vw;
    if (s.SS / vw % 2 == 0) s.SS += vw;
    s.threads = (N + 31) / 32 * 64;
    s.smem = (2 * 8 * (size_t)s.SS + 64) * elem;
    s.ok = N >= 2 && s.KC > 0 && (elem == 4 ? N <= 256 : N <= 128);
    return s;
}

template <class T, int KC, int WAVES>
static void launch_block_w(const T* SC, const SimArgs& a, const BlockShape& s, hipStream_t st) {
    constexpr int MAXT = KC <= 16 ? 256 : 512;
    hipLaunchKernelGGL((k_sim_block<T, 4, KC, MAXT, WAVES>), dim3(a.B), dim3(s.threads), s.smem, st, SC, a, s.SS);
}

// Registers against waves (FP32, N <= 128).  With few simulations a CU the
// substep's latency counts, with many the waves that hide it: the build for four
// waves a SIMD (128 VGPRs, what is used once a millisecond spilled) against the
// one without spills takes, in cycles a substep, N = 41: 527 / 537 at 128
// simulations, 1097 / 1403 at 2048; N = 64: 555 / 575 and 1195 / 1488; N = 100:
// 698 / 677, 844 / 822 at 512, 1436 / 1602 at 1024, 2657 / 3068 at 2048.
// Where the population (N <= 64) comes to more than half of a second or third wave a
// SIMD, a build that leaves no room for another: behind other kernels the dispatcher has
// put one more on some SIMDs and one less on others.  300 ms of 64 nodes, 769 / 900 / 1024
// simulations behind the analytical FIC: 1.22 / 1.25 / 1.27 ms, 0.93 / 0.95 / 0.99 with
// it (E/I kernel: 1.02 / 1.03 / 1.05); 32 nodes, 3000: 1.29, 1.07
// (1.10).  Where the deal is even it costs up to 3 %.
template <class T, int KC>
static void launch_block(const T* SC, const SimArgs& a, const BlockShape& s, hipStream_t st) {
    if constexpr (sizeof(T) == 4 && KC <= 8) {
        const int waves = a.B * (s.threads / 64), per = (waves + 1023) / 1024;   // per SIMD
        if (2 * waves > 2048 * per - 1024 && (per == 2 || per == 3)) {
            if (per == 2) hipLaunchKernelGGL((k_sim_block_most<T, 4, KC, 128, 2>), dim3(a.B), dim3(s.threads), s.smem, st, SC, a, s.SS);
            else hipLaunchKernelGGL((k_sim_block_most<T, 4, KC, 128, 3>), dim3(a.B), dim3(s.threads), s.smem, st, SC, a, s.SS);
            return;
        }
    }
    if constexpr (sizeof(T) == 4 && KC <= 8) {
        launch_block_w<T, KC, 4>(SC, a, s, st);
    } else if constexpr (sizeof(T) == 4 && KC <= 16) {
        if (a.B > 512) launch_block_w<T, KC, 4>(SC, a, s, st);
        else launch_block_w<T, KC, 1>(SC, a, s, st);
    } else {
        launch_block_w<T, KC, 1>(SC, a, s, st);
    }
}

template <class T>
hipError_t launch_sim_block(const T* SC, const SimArgs& a, hipStream_t st) {
    const BlockShape s = block_shape(a.N, sizeof(T));
    if (!s.ok) return hipErrorInvalidValue;
    switch (s.KC) {
        case 4: launch_block<T, 4>(SC, a, s, st); break;
        case 6: launch_block<T, 6>(SC, a, s, st); break;
        case 8: launch_block<T, 8>(SC, a, s, st); break;
        case 10: launch_block<T, 10>(SC, a, s, st); break;
        case 13: launch_block<T, 13>(SC, a, s, st); break;
        case 16: launch_block<T, 16>(SC, a, s, st); break;
        default:
            if constexpr (sizeof(T) == 4) {
                switch (s.KC) {
                    case 20: launch_block<T, 20>(SC, a, s, st); break;
                    case 25: launch_block<T, 25>(SC, a, s, st); break;
                    case 28: launch_block<T, 28>(SC, a, s, st); break;
                    default: launch_block<T, 32>(SC, a, s, st); break;
                }
                break;
            }
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template hipError_t launch_sim_block<float>(const float*, const SimArgs&, hipStream_t);
template hipError_t launch_sim_block<double>(const double*, const SimArgs&, hipStream_t);

}  // namespace bnm
