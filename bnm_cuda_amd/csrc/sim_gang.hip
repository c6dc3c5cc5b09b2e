// sim_gang.hip -- integration kernel for node counts whose SC one CU does not
// hold: a simulation runs on C workgroups ("members"), each with the rows of SC
// and the updates of its own nodes, that exchange S_E every substep.
//
// Layout of a member: four waves of 4 groups of 16 lanes; a group holds R nodes
// and all of k in 16 slices of KC values, so a lane keeps R x KC values of SC in
// VGPRs.  The sums over the 16 slices are DPP adds within the group (cf.
// k_sim_block); every node's sum ends up in 16 / R lanes, even lanes step the
// excitatory pool, odd ones the inhibitory (the lanes past the first two of a
// node repeat them and write nothing).
//
// Exchange: one 64-bit word per node (FP32; two for FP64, 32 bits each) holds
// the new S_E and the number of its substep: a word is its own flag, so no
// fence is needed.  A poll reads two words (16 bytes), each checked by itself.
// The members of a simulation get block indices 8 apart, i.e. one XCD, and meet in
// its L2: a plain store (the L1 writes through) is seen by a
// poll that passes the L1 by (agent scope) 0.27 us later; a store of agent scope
// goes on to memory and takes 0.39 us.  That the members do share an XCD is
// checked when they start.  Words are double-buffered by substep parity; a
// member that writes substep n + 2 has read every other member's n + 1, which
// they wrote after reading all of n.  Four more waves do the polling, one beside
// each wave that computes: loads return in order, so a wave that polls would
// wait for its noise from HBM first.
//
// Waiting: members start when all are there and on one XCD.  A member that waits
// in vain (GangArgs::start_polls, 1.6 s: another kernel holds the CUs) marks the
// simulation, and tells the rest of the launch, whose members then wait no more: those
// that do not find all the others there mark at once, so a launch waits once.  It waits
// that long because the CUs mostly come free: two contexts of 32 simulations of N = 400,
// FP32, each 0.155 s by itself, run at the same time take 0.31 s (0.60 s with a wait of
// 33 ms for each simulation).  Every member of a marked simulation ends, and the launch that
// follows in the stream (k_sim_gang_alone) runs the marked simulations on one
// workgroup each, with the members' arithmetic: a simulation's results do not depend on
// whether its members met.  From then on all members are resident, and the polls in the
// time loop end when the others get there; they have a bound too (kLoopPolls),
// with the same consequence.  A group of members runs one simulation after the other,
// as many groups as have a CU for each member: members of a second round of
// workgroups would start one by one, as simulations of the first end, and wait in
// vain for each other (FP64, 128 simulations of N = 400 with FIC, 2.7 s: 0.64 s with
// the hybrid kernel behind them, 0.48 on that alone, 0.22 with groups).
//
// What bounds it: the exchange.  At N = 400 (FP32, 16 simulations on 112 CUs) one
// substep is 1810 cycles: 850 from store to the value in the others' LDS, 450 of
// FMAs (100 a lane) and LDS reads, 160 of update, the rest sums, barrier and BW;
// the sparse kernel on one CU, which walks its row with an add, a gather and an
// FMA per nonzero, takes 6330 (40 % dense).  FP64, N = 200 (32 simulations on 128
// CUs): 2030 against the sparse kernel's 3020 (33 % dense) and the hybrid's 11660.
// Polling with two loads in flight, or with pauses, is no faster (1980, 1760 to
// 1880 cycles).  LDS-resident S has to be 16-byte aligned: behind the three
// flags without it every 16-byte read took several times as long (3060 cycles).
#include <algorithm>
#include <type_traits>

#include "kernels.hpp"
#include "model.hpp"
#include "pool.hpp"

namespace bnm {

namespace {

constexpr int kRor4 = 0x124, kRor8 = 0x128;
constexpr int kLoopPolls = 1 << 22;    // x ~0.4 us

typedef unsigned long long u64;
constexpr u64 kGangAbort = 1ull << 63;
constexpr int kDropped = 0x40000000;   // lane offset beyond the exchange words: the access is dropped
constexpr int kSc1 = 0x10;             // cache policy of a load that passes the L1 by

__device__ __forceinline__ u64 xload(const u64* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void xstore(u64* p, unsigned seq, unsigned v) {
    __hip_atomic_store(p, ((u64)seq << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Sum of acc over the 16 lanes of a group for the lane's own node.  acc[r] of
// lane q belongs to node n ^ r (R = 2), n, n ^ 1, 3 - n, (3 - n) ^ 1 (R = 4),
// n = gang_node(q): a lane keeps its own half of the rows and takes its mirror
// image's sums of them.
template <int R>
__device__ __forceinline__ int gang_node(int q) { return (q & (2 * R - 1)) >> 1; }
template <int R>
__device__ __forceinline__ int gang_row(int q, int r) {
    const int n = gang_node<R>(q);
    return ((r & 2) ? 3 - n : n) ^ (r & 1);
}
template <class T>
__device__ __forceinline__ T gang_sum(T (&acc)[4]) {
    T a0 = acc[0] + dpp<kMirror16>(acc[2]), a1 = acc[1] + dpp<kMirror16>(acc[3]);
    a0 += dpp<kRor8>(a0);
    a1 += dpp<kRor8>(a1);
    const T c = a0 + dpp<kXor2>(a1);
    return c + dpp<kXor1>(c);
}
template <class T>
__device__ __forceinline__ T gang_sum(T (&acc)[2]) {
    T a0 = acc[0] + dpp<kRor8>(acc[0]), a1 = acc[1] + dpp<kRor8>(acc[1]);
    a0 += dpp<kRor4>(a0);
    a1 += dpp<kRor4>(a1);
    const T c = a0 + dpp<kXor2>(a1);
    return c + dpp<kXor1>(c);
}

}  // namespace

// one simulation on the C workgroups of a group; every thread of a member returns
// after the same number of barriers
template <class T, int R, int KC>
__device__ __forceinline__ void gang_run(const T* __restrict__ SC, const SimArgs& a, const GangArgs& ga, int SS,
                                         int member, int sim) {
    constexpr bool F64 = sizeof(T) == 8;
    constexpr int WPV = sizeof(T) / 4;             // exchange words per node
    constexpr int NPU = 2 / WPV;                    // nodes in the 16 bytes of a poll
    constexpr int PU = F64 && R == 2 ? 2 : 1;      // polls of a thread
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    constexpr int VW = 16 / sizeof(T);
    typedef T vec __attribute__((ext_vector_type(VW)));
    const int C = ga.C;
    const int N = a.N, tid = threadIdx.x & 255, threads = kGangThreads;
    const bool poller = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) != 0;
    const int lane = tid & 63, q = lane & 15, pop = lane & 1;
    constexpr int rows = 16 * R;                    // nodes of a member
    const int base = member * rows, mine = min(rows, N - base);
    const int j0 = base + (tid >> 4) * R;           // the group's first node
    const int j = j0 + gang_node<R>(q);
    const bool comp = !poller && j < N && q < 2 * R;   // (the lanes that write)
    const bool writer = comp && pop == 0;
    const int jc = min(j, N - 1);
    const int ldS = 16 * SS;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* Sb = reinterpret_cast<T*>(smem_raw);         // [2][ldS], then slots nobody reads
    __shared__ int dead, vote, votes;               // given up; out of band here, anywhere
    u64* state = ga.state + sim;
    if (threadIdx.x == 0) {
        // all members present and on one XCD, or none runs: the low byte counts
        // the members, five bits per XCD those on it
        unsigned xcc;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
        const int sh = 8 + 5 * (int)(xcc & 7);
        int d = 0;
        __hip_atomic_fetch_add(state, 1ull + (1ull << sh), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int n = 0;; ++n) {
            u64 v = xload(state);
            if (v & kGangAbort) { d = 1; break; }
            const bool all = (int)(v & 255) >= C;
            if (all && (int)((v >> sh) & 31) == C) break;
            if (!all && n >= ga.start_polls)
                __hip_atomic_store(ga.gave_up, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((all || xload(ga.gave_up)) &&
                __hip_atomic_compare_exchange_strong(state, &v, v | kGangAbort, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT)) {
                d = 1;
                break;
            }
            __builtin_amdgcn_s_sleep(4);
        }
        dead = d;
        vote = votes = 0;
    }
    for (int i = threadIdx.x; i < 2 * ldS; i += threads) {
        const int slot = i % ldS, qq = slot % SS, k = (slot / SS) * KC + qq;
        Sb[i] = (qq < KC && k < N) ? T(0.001) : T(0);
    }
    const T* Sr = Sb + q * SS;
    auto place = [&](int k) { return (k / KC) * SS + k % KC; };
    const int own = writer ? place(j) : 2 * ldS + lane;   // (buffer 1: + ldS for writers)
    const int own1 = writer ? own + ldS : own;
    // exchange words [parity][units of 16 bytes]
    const int units = (N + NPU - 1) / NPU, xrow = units * 16;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        ga.xch + (size_t)sim * units * 4, (short)0, 2 * xrow, 0x00020000);
    u64* xflag = ga.flag + (size_t)sim * kGangMembers;
    int ts = 0, trial = 0;
    unsigned seq = 0;
    bool adjusting = a.adjust_fic != 0;
    __syncthreads();
    if (dead) return;

    if (poller) {
        // the units of the others that this thread waits for, and where they go
        // (a thread without one repeats the first and keeps nothing)
        const int u0 = base / NPU, um = (mine + NPU - 1) / NPU, other = units - um;
        int px[PU], pl[PU][NPU];
        bool two[PU];                               // the unit's second word is a node's
#pragma unroll
        for (int w = 0; w < PU; ++w) {
            const int i = tid + w * 256, e = i < other ? i : 0, u = e < u0 ? e : e + um;
            px[w] = u * 16;
            two[w] = F64 || 2 * u + 1 < N;
#pragma unroll
            for (int h = 0; h < NPU; ++h) {
                const int k = u * NPU + h;
                pl[w][h] = (i < other && k < N) ? place(k) : 2 * ldS + lane;
            }
        }
        while (ts <= a.time_steps) {
            for (int s = 0; s < 10; ++s) {
                const int xo = ((s + 1) & 1) * xrow;
                ++seq;
                u32x4 x[PU];
                for (int n = 0;; ++n) {
                    bool all = true;
#pragma unroll
                    for (int w = 0; w < PU; ++w) x[w] = __builtin_amdgcn_raw_buffer_load_b128(xr, px[w], xo, kSc1);
#pragma unroll
                    for (int w = 0; w < PU; ++w) all = all && x[w][1] == seq && (x[w][3] == seq || !two[w]);
                    if (__all(all)) break;
                    asm volatile("" ::: "memory");
                    if ((n & 1023) == 1023 && (n > kLoopPolls || *(volatile int*)&dead)) {
                        dead = 1;
                        break;
                    }
                }
                T* Sw = Sb + ((s & 1) ? 0 : ldS);
#pragma unroll
                for (int w = 0; w < PU; ++w) {
                    if constexpr (F64) {
                        Sw[pl[w][0]] = __longlong_as_double(((u64)x[w][2] << 32) | x[w][0]);
                    } else {
                        Sw[pl[w][0]] = __uint_as_float(x[w][0]);
                        Sw[pl[w][NPU - 1]] = __uint_as_float(x[w][2]);
                    }
                }
                lds_barrier();
            }
            if (dead) return;
            ++ts;
            if (adjusting && ts == a.i_end) {
                lds_barrier();
                lds_barrier();
                adjusting = votes != 0 && trial < a.max_fic_trials;
                if (adjusting) {
                    ts = 0;
                    ++trial;
                }
                lds_barrier();
            }
        }
        return;
    }

    const int xput = writer ? j * 8 * WPV : kDropped;
    T sc[R][KC];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int row = j0 + gang_row<R>(q, r);
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            const int k = q * KC + i;
            sc[r][i] = (row < N && k < N) ? SC[(size_t)row * N + k] : T(0);
        }
    }
    const size_t o = (size_t)sim * N + jc;
    Pool<T> p;
    p.init(pop, a.G[sim], a.wEE[o], a.wEI[o], a.wIE_in[o]);
    double delta = a.init_delta;
    // FP32: BW in parts, a millisecond behind; FP64: the reference's order at
    // the end of the millisecond
    typename std::conditional<F64, BW<double>, BWParts<float>>::type bw;
    bw.reset();
    T bwS = 0;
    int bold_vol = -1;
    double mI = 0, ext[3] = {0, 0, 0};
    int vol = 0, next_vol = 0;
    bool failed = false;
    const unsigned dur = (unsigned)(a.i_end - a.i_start + 1);
    const int P = (int)a.noise_period;
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
    int ms1 = P > 1 ? 1 : 0;
#pragma unroll
    for (int s = 0; s < 10; ++s) nz[s] = draw(0, s);
    p.before(nz[0]);
    nz[0] = draw(ms1, 0);
    while (ts <= a.time_steps) {
        const int ms2 = ms1 + 1 == P ? 0 : ms1 + 1;
#pragma unroll
        for (int s = 0; s < 10; ++s) {
            ++seq;
            // the next millisecond's draw, ahead of the store that the others wait for
            // (behind it: 2030 cycles a substep against 1810)
            const float drawn = s < 9 ? draw(ms1, s + 1) : draw(ms2, 0);
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
            T acc[R];
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r] = sc[r][0] * v[0];
#pragma unroll
            for (int i = 1; i < KC; ++i)
#pragma unroll
                for (int r = 0; r < R; ++r) acc[r] = fma(sc[r][i], v[i], acc[r]);
            const T c = gang_sum(acc);
            p.after(c, s == 9);
            if constexpr (F64) {
                const u64 u = __double_as_longlong(p.S);
                __builtin_amdgcn_raw_buffer_store_b128(u32x4{(unsigned)u, seq, (unsigned)(u >> 32), seq}, xr, xput,
                                                       ((s + 1) & 1) * xrow, 0);
            } else {
                __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(p.S), seq}, xr, xput,
                                                      ((s + 1) & 1) * xrow, 0);
            }
            Sb[(s & 1) ? own : own1] = p.S;
            // while the words are on their way
            p.settle();
            if (s < 9) {
                p.before(nz[s + 1]);
                nz[s + 1] = drawn;
            } else {
                p.before(nz[0]);
                nz[0] = drawn;
            }
            if constexpr (F64) {
                if (s == 9 && writer) bw.step(p.S);
            } else {
                if (s == 1) bw.template part<0>(bwS);
                if (s == 2) bw.template part<1>(bwS);
                if (s == 3) bw.template part<2>(bwS);
                if (s == 4) bw.template part<3>(bwS);
                if (s == 5) bw.template part<4>(bwS);
                if (s == 6) bw.template part<5>(bwS);
            }
            lds_barrier();
        }
        if (dead) {
            if (threadIdx.x == 0) __hip_atomic_fetch_or(state, kGangAbort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        ms1 = ms2;
        if constexpr (!F64) {
            if (bold_vol >= 0) store_bold(bold_vol);
            bold_vol = -1;
            bwS = p.S;
        }
        if (ts == next_vol) {
            next_vol += a.bold_tr;
            if constexpr (F64) store_bold(vol);
            else bold_vol = vol;
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
                // out of band in any member: each publishes its own answer under
                // the number of the last substep and waits for the others'
                const bool out = writer && fic_decide<double>(mI, dur, trial, a.max_fic_trials, p.wIE, delta);
                p.set_wIE(pop == 0);
                if (out) vote = 1;
                lds_barrier();
                if (threadIdx.x == 0) xstore(xflag + member, seq, vote ? 1u : 0u);
                if ((int)threadIdx.x < C) {
                    u64 w;
                    for (int n = 0;; ++n) {
                        w = xload(xflag + tid);
                        if ((unsigned)(w >> 32) == seq) break;
                        if ((n & 1023) == 1023 && (n > kLoopPolls || *(volatile int*)&dead)) {
                            dead = 1;
                            break;
                        }
                    }
                    if ((unsigned)w != 0) votes = 1;
                }
                lds_barrier();
                if (votes) {
                    if (trial < a.max_fic_trials) {
                        p.reset();
                        bw.reset();
                        bwS = 0;
                        bold_vol = -1;
                        mI = 0;
                        ext[0] = ext[1] = ext[2] = 0;
                        for (int k = tid; k < N; k += 256) Sb[place(k)] = T(0.001);
                        ts = 0; vol = 0; next_vol = 0; ++trial;
                        ms1 = P > 1 ? 1 : 0;
#pragma unroll
                        for (int s = 0; s < 10; ++s) nz[s] = draw(0, s);
                        p.before(nz[0]);
                        nz[0] = draw(ms1, 0);
                    } else {
                        failed = true; adjusting = false;
                    }
                } else {
                    adjusting = false;
                }
                lds_barrier();
                if (threadIdx.x == 0) vote = votes = 0;
            }
        }
    }
    if (dead) {                                     // (in the FIC's exchange of the last millisecond)
        if (threadIdx.x == 0) __hip_atomic_fetch_or(state, kGangAbort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    if constexpr (!F64) {
        bw.template part<0>(bwS);
        bw.template part<1>(bwS);
        bw.template part<2>(bwS);
        bw.template part<3>(bwS);
        bw.template part<4>(bwS);
        bw.template part<5>(bwS);
        if (bold_vol >= 0) store_bold(bold_vol);
    }
    if (comp) {
        if (pop == 0) a.wIE_out[o] = p.wIE;
        const int n = vol - a.n_vols_remove;
        for (int i = 0; i < 3; ++i) a.ext[((size_t)sim * 6 + 3 * pop + i) * N + j] = n > 0 ? ext[i] / n : 0.0;
    }
    if (member == 0 && threadIdx.x == 0) {
        a.fic_failed[sim] = failed ? 1 : 0;
        a.fic_trials[sim] = trial;
    }
}

// A group of members takes one simulation after the other, so that all members are
// resident from the start, whatever the population: a workgroup a CU.
template <class T, int R, int KC>
__global__ __launch_bounds__(kGangThreads) void k_sim_gang(const T* __restrict__ SC, SimArgs a, GangArgs ga, int SS) {
    const int member = (blockIdx.x >> 3) % ga.C;
    if (member >= ga.present) return;
    for (int sim = (blockIdx.x >> 3) / ga.C * 8 + (blockIdx.x & 7); sim < a.B; sim += 8 * ga.groups) {
        gang_run<T, R, KC>(SC, a, ga, SS, member, sim);
        __syncthreads();
    }
}

// The simulations that are marked, one workgroup each, with the bits of gang_run: a
// node's sum is that of 16 slices of KC values, each an FMA chain in order of k, added
// in gang_sum's tree.  That is, with s_q the sum of slice q, (T_0 + T_2) + (T_1 + T_3),
// R = 4: T_i = (s_i + s_15-i) + (s_i+8 + s_7-i), R = 2: (s_i + s_i+8) + (s_i+4 + s_i+12).
// A lane sums slices of one node, with SC streamed column by column from L2: KS waves a
// node, one T_i each, or two.  Then a lane steps one pool.  Bound by that stream: N = 400,
// FP32, 11 us a substep, FP64 21.
template <class T, int R, int KC>
__global__ __launch_bounds__(1024) void k_sim_gang_alone(const T* __restrict__ SCt, SimArgs a, const u64* __restrict__ state,
                                                         int KS) {
    constexpr bool F64 = sizeof(T) == 8;
    const int sim = blockIdx.x;
    if (!(state[sim] & kGangAbort)) return;
    const int N = a.N, NW = (N + 63) / 64, tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = wave % NW, ks = wave / NW;
    const int col = nw * 64 + lane, colc = min(col, N - 1);          // the node that this lane sums for
    const int pop = tid & 1, j = tid >> 1, jc = min(j, N - 1);        // the pool that it steps
    const bool comp = j < N, writer = comp && pop == 0, steps = wave * 32 < N;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    constexpr int ldS = 16 * KC;                    // (S_E past the last node is 0, and so is SCt)
    T* Sb = reinterpret_cast<T*>(smem_raw);         // [2][ldS]
    T* part = Sb + 2 * ldS;                         // [KS][64 NW]
    const __amdgpu_buffer_rsrc_t scr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(SCt), (short)0, (N + (int)kSCtPad) * N * (int)sizeof(T), 0x00020000);
    const int voff = colc * (int)sizeof(T);
    auto column = [&](int k) __attribute__((always_inline)) {             // SC[the lane's node][k]
        const int so = k * N * (int)sizeof(T);
        if constexpr (F64) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(scr, voff, so, 0);
            return __longlong_as_double(((long long)v[1] << 32) | v[0]);
        } else {
            return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(scr, voff, so, 0));
        }
    };
    auto four = [&](const T* S, int i) __attribute__((always_inline)) {   // T_i
        const int sl[4] = {i, R == 4 ? 15 - i : i + 8, R == 4 ? i + 8 : i + 4, R == 4 ? 7 - i : i + 12};
        constexpr int U = 4;                        // (x 4 loads on the way together)
        T s[4] = {T(0), T(0), T(0), T(0)};
        auto batch = [&](auto n, int m0) __attribute__((always_inline)) {
            constexpr int M = decltype(n)::value;
            T w[M][4];
#pragma unroll
            for (int u = 0; u < M; ++u)
#pragma unroll
                for (int q = 0; q < 4; ++q) w[u][q] = column(sl[q] * KC + m0 + u);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < M; ++u)
#pragma unroll
                for (int q = 0; q < 4; ++q) s[q] = fma(w[u][q], S[sl[q] * KC + m0 + u], s[q]);
        };
#pragma unroll 1
        for (int m0 = 0; m0 + U <= KC; m0 += U) batch(std::integral_constant<int, U>{}, m0);
        if constexpr (KC % U != 0) batch(std::integral_constant<int, KC % U>{}, KC / U * U);
        return (s[0] + s[1]) + (s[2] + s[3]);
    };
    for (int i = tid; i < 2 * ldS; i += blockDim.x) Sb[i] = i % ldS < N ? T(0.001) : T(0);
    const size_t o = (size_t)sim * N + jc;
    Pool<T> p;
    p.init(pop, a.G[sim], a.wEE[o], a.wEI[o], a.wIE_in[o]);
    double delta = a.init_delta;
    typename std::conditional<F64, BW<double>, BWParts<float>>::type bw;
    bw.reset();
    double mI = 0, ext[3] = {0, 0, 0};
    int ts = 0, vol = 0, trial = 0;
    bool adjusting = a.adjust_fic != 0, failed = false;
    const unsigned dur = (unsigned)(a.i_end - a.i_start + 1);
    const int P = (int)a.noise_period;
    auto draw = [&](int ms, int s) { return a.noise[(((size_t)ms * 10 + s) * N + jc) * 2 + pop]; };
    p.before(draw(0, 0));
    __syncthreads();
    while (ts <= a.time_steps) {
        const int ms = ts % P, ms1 = ms + 1 == P ? 0 : ms + 1;
#pragma unroll 1
        for (int s = 0; s < 10; ++s) {
            const T* S = Sb + (s & 1) * ldS;
            const float drawn = s < 9 ? draw(ms, s + 1) : draw(ms1, 0);
            part[ks * 64 * NW + col] = KS == 4 ? four(S, ks) : four(S, ks) + four(S, ks + 2);
            __syncthreads();
            if (steps) {
                const T* c = part + jc;
                const int ld = 64 * NW;
                p.after(KS == 4 ? (c[0] + c[2 * ld]) + (c[ld] + c[3 * ld]) : c[0] + c[ld], s == 9);
                if (writer) Sb[((s + 1) & 1) * ldS + j] = p.S;
                p.settle();
                p.before(drawn);
            }
            __syncthreads();
        }
        if constexpr (F64) {
            bw.step(p.S);
        } else {
            bw.template part<0>(p.S);
            bw.template part<1>(p.S);
            bw.template part<2>(p.S);
            bw.template part<3>(p.S);
            bw.template part<4>(p.S);
            bw.template part<5>(p.S);
        }
        if (ts % a.bold_tr == 0) {
            if (writer)
                reinterpret_cast<T*>(a.bold)[((size_t)sim * a.output_ts + vol) * N + j] =
                    (T)bw.bold(a.bw_k1, a.bw_k2, a.bw_k3);
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
                const bool out = writer && fic_decide<double>(mI, dur, trial, a.max_fic_trials, p.wIE, delta);
                p.set_wIE(pop == 0);
                if (!__syncthreads_or(out)) {
                    adjusting = false;
                } else if (trial < a.max_fic_trials) {
                    p.reset();
                    bw.reset();
                    mI = 0;
                    ext[0] = ext[1] = ext[2] = 0;
                    if (writer) Sb[j] = p.S;
                    ts = 0; vol = 0; ++trial;
                    p.before(draw(0, 0));
                    __syncthreads();
                } else {
                    failed = true; adjusting = false;
                }
            }
        }
    }
    if (comp) {
        if (pop == 0) a.wIE_out[o] = p.wIE;
        const int n = vol - a.n_vols_remove;
        for (int i = 0; i < 3; ++i) a.ext[((size_t)sim * 6 + 3 * pop + i) * N + j] = n > 0 ? ext[i] / n : 0.0;
    }
    if (tid == 0) {
        a.fic_failed[sim] = failed ? 1 : 0;
        a.fic_trials[sim] = trial;
    }
}

// marks every n-th simulation before any member looks
__global__ void k_gang_mark(u64* state, int B, int n) {
    for (int i = threadIdx.x * n; i < B; i += blockDim.x * n) state[i] = kGangAbort;
}

// FP32: N of 257 to 512, R = 4 (64 nodes a member).  FP64: 129 to 256 with R = 4,
// to 512 with R = 2 (32 nodes a member: R x KC doubles are the same VGPRs).
static const int kGangKC[] = {10, 13, 16, 20, 25, 28, 32};

GangShape gang_shape(int N, size_t elem) {
    GangShape s{};
    s.R = elem == 4 || N <= 256 ? 4 : 2;
    const int per = (N + 15) / 16;
    for (int kc : kGangKC)
        if (kc >= per) { s.KC = kc; break; }
    const int vw = 16 / (int)elem;
    s.SS = (s.KC + vw - 1) / vw * vw;
    if (s.SS / vw % 2 == 0) s.SS += vw;
    s.C = (N + 16 * s.R - 1) / (16 * s.R);
    s.smem = (3 * 16 * (size_t)s.SS + 64) * elem;
    s.ok = s.KC > 0 && s.C <= kGangMembers && (elem == 4 ? N > 256 : N > 128) && N <= 512;
    return s;
}

// (a row of FP32 words is rounded up to whole 16-byte units)
static size_t gang_row_words(int N, size_t elem) { return elem == 4 ? ((size_t)N + 1) / 2 * 2 : 2 * (size_t)N; }

size_t gang_words(int N, int B, size_t elem) {
    return (size_t)B * (gang_row_words(N, elem) * 2 + kGangMembers + 1) + 1;
}

template <class T, int R, int KC>
static void launch_gang(const T* SC, const T* SCt, const SimArgs& a, const GangArgs& g, const GangShape& s, hipStream_t st) {
    hipLaunchKernelGGL((k_sim_gang<T, R, KC>), dim3(8 * s.C * g.groups), dim3(kGangThreads), s.smem, st, SC, a,
                       g, s.SS);
    const int NW = (a.N + 63) / 64, KS = NW <= 4 ? 4 : 2;
    const size_t smem = (2 * 16 * KC + KS * 64 * (size_t)NW) * sizeof(T);
    hipLaunchKernelGGL((k_sim_gang_alone<T, R, KC>), dim3(a.B), dim3(KS * 64 * NW), smem, st, SCt, a, g.state, KS);
}

template <class T>
hipError_t launch_sim_gang(const T* SC, const T* SCt, const SimArgs& a, unsigned long long* words, int start_polls,
                           int mark, int cus, hipStream_t st) {
    const GangShape s = gang_shape(a.N, sizeof(T));
    if (!s.ok) return hipErrorInvalidValue;
    GangArgs g{};
    g.C = s.C;
    g.start_polls = start_polls;
    g.xch = words;
    g.groups = std::max(1, std::min((a.B + 7) / 8, cus / 8 / s.C));   // per XCD
    g.flag = words + (size_t)a.B * 2 * gang_row_words(a.N, sizeof(T));
    g.state = g.flag + (size_t)a.B * kGangMembers;
    g.gave_up = g.state + a.B;
    g.present = mark < 0 ? s.C - 1 : s.C;
    // no word carries a number yet, no member is there, no simulation is marked
    hipError_t e = launch_fill_i32(reinterpret_cast<int*>(words), (long long)gang_words(a.N, a.B, sizeof(T)) * 2, 0, st);
    if (e != hipSuccess) return e;
    if (mark > 0) hipLaunchKernelGGL(k_gang_mark, dim3(1), dim3(256), 0, st, g.state, a.B, mark);
    switch (s.KC) {
        case 10: if constexpr (sizeof(T) == 8) launch_gang<T, 4, 10>(SC, SCt, a, g, s, st); break;
        case 13: if constexpr (sizeof(T) == 8) launch_gang<T, 4, 13>(SC, SCt, a, g, s, st); break;
        case 16: if constexpr (sizeof(T) == 8) launch_gang<T, 4, 16>(SC, SCt, a, g, s, st); break;
        case 20: launch_gang<T, sizeof(T) == 4 ? 4 : 2, 20>(SC, SCt, a, g, s, st); break;
        case 25: launch_gang<T, sizeof(T) == 4 ? 4 : 2, 25>(SC, SCt, a, g, s, st); break;
        case 28: launch_gang<T, sizeof(T) == 4 ? 4 : 2, 28>(SC, SCt, a, g, s, st); break;
        default: launch_gang<T, sizeof(T) == 4 ? 4 : 2, 32>(SC, SCt, a, g, s, st); break;
    }
    return hipGetLastError();
}

const unsigned long long* gang_state(const unsigned long long* words, int N, int B, size_t elem) {
    return words + (size_t)B * (2 * gang_row_words(N, elem) + kGangMembers);
}

template hipError_t launch_sim_gang<float>(const float*, const float*, const SimArgs&, unsigned long long*, int, int, int,
                                           hipStream_t);
template hipError_t launch_sim_gang<double>(const double*, const double*, const SimArgs&, unsigned long long*, int, int,
                                            int, hipStream_t);

}  // namespace bnm
