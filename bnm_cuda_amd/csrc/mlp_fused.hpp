// mlp_fused.hpp -- training and prediction of networks whose layers are at most
// 256 wide, in three launches a step (mlp.hip includes it).
//
//  k_mlp     one workgroup takes 8 to 32 rows through all layers, forward and, for
//            a gradient, back again: the activations stay in LDS, the weights come
//            from L2 as MFMA fragments (16 bytes a lane, no staging).  It leaves
//            dZ and, as fragments for products over the rows, the activations and
//            dZ once more.
//  k_mlp_dw  the weight gradients of all layers (dW = dZ^T A, 64 x 64 tiles, split
//            over the rows) straight from those fragments, and the bias gradients
//            (column sums of dZ).
//  k_mlp_fin sums the row splits and, in training, steps Adam and rewrites the
//            weights' operand copies.
//
// What bounded a step before (4 x 256 hidden, 1024 rows, BF16): 28 launches of 4
// to 35 us in sequence, each GEMM waiting for a 32-deep K chunk to arrive, be
// rounded and be staged in LDS before the next was asked for; 450 us for 0.4
// GFLOP.  Now 45 us: 27 + 7 + 6 us and the gaps.  The products are the same MFMAs
// in the same order of k, rows are split over the same ranges, and the splits and
// column sums are added in the same order, so gradients and steps are the same
// bits.
#pragma once

namespace {

constexpr int kFusedDim = 256, kFusedLayers = 16;

template <bool BF16> struct Op;   // operand type of the products
template <> struct Op<true> {
    typedef unsigned short E;
    typedef u16x8 frag;
    static constexpr int KS = 32, EPV = 8;   // k per step, per lane fragment
    static __device__ __forceinline__ int at(int k) { return k; }   // where k lies among the operand's values
    static __device__ __forceinline__ E make(float v) { return f2bf(v); }
    static __device__ __forceinline__ f32x4 mma(frag a, frag b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    }
};
template <> struct Op<false> {
    typedef float E;
    typedef f32x4 frag;
    static constexpr int KS = 16, EPV = 4;
    static __device__ __forceinline__ E make(float v) { return v; }
    // a lane's four values are those of four MFMAs in turn: k = 16 step + 4 s + lane / 16
    static __device__ __forceinline__ int at(int k) { return (k & ~15) | (k & 3) << 2 | (k >> 2 & 3); }
    static __device__ __forceinline__ f32x4 mma(frag a, frag b, f32x4 c) {
#pragma unroll
        for (int s = 0; s < 4; ++s) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], c, 0, 0, 0);
        return c;
    }
};

struct FusedLayer {
    int K, N;
    const void *Wf, *Wb;   // operand copies: W by column (n) tiles and by row (k) tiles, zero padded
    const float* b;
    float* G;              // gelu'(Z): [workgroups][tiles][threads][4], each thread's own
    float* dZ;             // [rows / 4][N][4]
    void *AT, *dT;         // input activations by k, dZ by n: operands that contract over rows
    float* part;           // [kz][N * K] weight gradient, one per row split
    int woff, boff;
};

struct FusedNet {
    const FusedLayer* l;   // on the device
    int L, rows, ldr;      // layers, rows, and rows padded to 32
    const float *X, *T;    // rows idx[0..rows) of X [*][in], T [*][out] (idx null: 0..rows)
    const int* idx;
    float* Y;              // prediction [rows][out]
    float* loss;           // [workgroups] partial sums of the loss
    const unsigned* W;     // all weights' operand copies
    unsigned wwords;
    float scale;
    int accum;             // add to loss
    int klen, kz;          // rows per split, splits
};

// A pointer read from the layer table, as one to device memory: the compiler
// would make flat accesses of it, which wait for LDS and each other.
template <class T> using Dev = T __attribute__((address_space(1)))*;
template <class T> __device__ __forceinline__ Dev<T> dev(const void* p) { return (Dev<T>)const_cast<void*>(p); }

// the layer table, read with scalar loads (kernels do not write it)
typedef const __attribute__((address_space(4))) FusedLayer ConstLayer;
__device__ __forceinline__ ConstLayer& layer_of(const FusedNet& n, int l) {
    return ((ConstLayer*)(__UINTPTR_TYPE__)n.l)[l];
}

__host__ __device__ inline int steps_of(int n, int per) { return (n + per - 1) / per; }

// Operand matrices lie fragment by fragment: tiles of 16 (i), within them steps
// of KS (k), within them the 64 lanes' EPV values, so that a wave's load is 1 KB
// in a row.  `steps` = steps of k.
template <bool BF16>
__device__ __forceinline__ size_t frag_at(int i, int k, int steps) {
    typedef Op<BF16> O;
    k = O::at(k);
    return ((size_t)((i >> 4) * steps + k / O::KS) * 64 + (k % O::KS) / O::EPV * 16 + (i & 15)) * O::EPV + k % O::EPV;
}

constexpr int kRowThreads = 512;    // 8 waves; wave w computes column tiles w and w + 8
constexpr int kStepsAhead = 8;      // k steps whose weights are loaded at a time

// Bound: latency.  1024 rows, 4 x 256 hidden, BF16, nine products: 55000 cycles, of
// which 6000 until the first (row indices, then rows, from memory), then each
// product 2200 (its workgroup reads 128 KB of weights at the 64 bytes a clock that
// a CU gets from L2) and its end 4100 forward (activation and derivative, stores)
// or 2200 back.  So the loads for the next eight steps of k, across products, go
// out before this step's products, and few rows go to a workgroup: with 8, both
// halves of an MFMA's 16 rows hold the same ones and the lanes' halves finish one
// of the wave's two column tiles each (16 rows: 38.7 us, 8: 36.4; all that is
// here: 27).
template <bool BF16, int ROWS, bool TRAIN>
__global__ __launch_bounds__(kRowThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_mlp(FusedNet n) {
    typedef Op<BF16> O;
    typedef typename O::E E;
    typedef typename O::frag frag;
    typedef E E4 __attribute__((ext_vector_type(4)));
    constexpr int R = ROWS, MT = (ROWS + 15) / 16, LD = kFusedDim + O::EPV, U = kStepsAhead;
    constexpr bool HALF = ROWS == 8;
    constexpr int NT = HALF ? 1 : 2;                        // column tiles that a lane finishes
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float red[kRowThreads / 64];
    E* const lds = reinterpret_cast<E*>(smem);
    auto act = [&](int i) { return lds + i * (R * LD); };   // two buffers
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c = lane & 15;
    const int row0 = blockIdx.x * R, rsteps = n.ldr / O::KS;
    const int total = TRAIN ? 2 * n.L - 1 : n.L;            // products: forward, then back to layer 1
    struct Prod {
        Dev<const frag> W;
        int K, N, nk, tiles;
    };
    auto product = [&](int s) __attribute__((always_inline)) {
        const bool fwd = s < n.L;
        ConstLayer& y = layer_of(n, fwd ? s : 2 * n.L - 1 - s);
        Prod p;
        p.W = dev<const frag>(fwd ? y.Wf : y.Wb);
        p.K = fwd ? y.K : y.N;
        p.N = fwd ? y.N : y.K;
        p.nk = steps_of(p.K, O::KS);
        p.tiles = steps_of(p.N, 16);
        return p;
    };
    // (steps and tiles past the last repeat it and are not used)
    auto load = [&](frag (&b)[U][2], const Prod& p, int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const Dev<const frag> W = p.W + (size_t)min(w + 8 * t, p.tiles - 1) * p.nk * 64 + lane;
#pragma unroll
            for (int u = 0; u < U; ++u) b[u][t] = W[min(k0 + u, p.nk - 1) * 64];
        }
    };
    // The weights were last written by the whole card, so each XCD's L2 has to
    // fetch them: its workgroups (every eighth) ask for their lines at once.
    unsigned line[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const unsigned o = ((i * ((gridDim.x + 7) >> 3) + (blockIdx.x >> 3)) * kRowThreads + tid) * 32;
        line[i] = n.W[min(o, n.wwords - 1)];
    }
    frag wa[U][2], wb[U][2];
    Prod p = product(0);
    load(wa, p, 0);
    const int rg = HALF ? 4 * (g & 1) : 4 * g;
    int src[MT][4];        // the rows that this lane finishes
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = min(row0 + 16 * m + rg + r, n.rows - 1);
            src[m][r] = TRAIN && n.idx ? n.idx[row] : row;
        }
    const float loss0 = TRAIN && n.accum && tid == 0 ? n.loss[blockIdx.x] : 0.0f;
    {
        const int K = layer_of(n, 0).K, Kp = p.nk * O::KS;
        const Dev<E> AT = dev<E>(layer_of(n, 0).AT);
        for (int e = tid; e < R * Kp; e += kRowThreads) {
            const int r = e / Kp, k = e % Kp, row = row0 + r;
            float v = 0.0f;
            if (row < n.rows && k < K) v = n.X[(size_t)(n.idx ? n.idx[row] : row) * K + k];
            act(0)[r * LD + O::at(k)] = O::make(v);
            if (TRAIN && k < K) AT[frag_at<BF16>(k, row, rsteps)] = O::make(v);
        }
    }
    // loads that are still out here would be waited for inside the loop, with its own
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(src[m][r]));
    bnm::lds_barrier();
    f32x4 acc[2][MT], gr[NT][MT];
    float s = 0.0f, bias[NT];
    const int half = HALF ? g >> 1 : 0;
    float want[NT][MT][4];
    auto tile = [&](int t) { return w + 8 * (HALF ? half : t); };
    auto own = [&](float* G, int t, int m) {
        return dev<f32x4>(G) + ((size_t)blockIdx.x * (NT * MT) + t * MT + m) * kRowThreads + tid;
    };
    int st = 0, k0 = 0, cur = 0;
    auto start = [&]() __attribute__((always_inline)) {   // of product st: what its end needs
        const bool fwd = st < n.L;
        ConstLayer& y = layer_of(n, fwd ? st : 2 * n.L - 2 - st);
#pragma unroll
        for (int t = 0; t < NT; ++t) bias[t] = dev<const float>(y.b)[min(16 * tile(t) + c, y.N - 1)];
        if (TRAIN && !fwd)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int m = 0; m < MT; ++m) gr[t][m] = *own(y.G, t, m);
        if (TRAIN && st == n.L - 1)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int m = 0; m < MT; ++m)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        want[t][m][r] = n.T[(size_t)src[m][r] * y.N + min(16 * tile(t) + c, y.N - 1)];
    };
    auto finish = [&]() __attribute__((always_inline)) {  // of product st: bias, activation or its derivative, and the operand of the next product
        const bool fwd = st < n.L, last = st == n.L - 1;
        ConstLayer& y = layer_of(n, fwd ? st : 2 * n.L - 2 - st);   // the layer whose Z or dZ it is
        const Dev<E> T = dev<E>(!TRAIN ? nullptr : fwd && !last ? layer_of(n, st + 1).AT : y.dT);
        E* out = act(cur ^ 1);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (tile(t) >= p.tiles) continue;
            const int col = 16 * tile(t) + c;
            const bool in = col < p.N;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int r0 = 16 * m + rg;
                float v[4] = {0, 0, 0, 0}, a[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) a[r] = HALF && half ? acc[1][m][r] : acc[t][m][r];
                if (fwd && !last) {
                    f32x4 d;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float z = a[r] + bias[t];
                        v[r] = in && row0 + r0 + r < n.rows ? gelu(z) : 0.0f;
                        d[r] = gelu_grad(z);
                    }
                    if (TRAIN) *own(y.G, t, m) = d;
                } else if (in) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = row0 + r0 + r;
                        if (row >= n.rows) continue;
                        if (!fwd) {
                            v[r] = a[r] * gr[t][m][r];
                        } else {
                            const float q = a[r] + bias[t];
                            if (TRAIN) {
                                const float d = q - want[t][m][r];
                                v[r] = 2.0f * d * n.scale;
                                s += d * d;
                            } else {
                                n.Y[(size_t)row * p.N + col] = q;
                            }
                        }
                    }
                }
                if (!TRAIN && last) continue;
                if (TRAIN && in && (last || !fwd))
                    dev<f32x4>(y.dZ)[(size_t)((row0 + r0) >> 2) * p.N + col] = f32x4{v[0], v[1], v[2], v[3]};
                E4 e;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    e[r] = O::make(v[r]);
                    out[(r0 + r) * LD + O::at(col)] = e[r];
                }
                if (TRAIN && in) {
                    if constexpr (BF16) {
                        *(Dev<E4>)(T + frag_at<BF16>(col, row0 + r0, rsteps)) = e;
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r) T[frag_at<BF16>(col, row0 + r0 + r, rsteps)] = e[r];
                    }
                }
            }
        }
        // columns between the last tile and the next product's last step
        if (steps_of(p.N, O::KS) * O::KS > p.tiles * 16 && tid < 16 * R)
            out[(tid >> 4) * LD + p.tiles * 16 + (tid & 15)] = O::make(0.0f);
        cur ^= 1;
        bnm::lds_barrier();
    };
    // eight steps of product st with weights b, after asking for the eight that follow in nx
    auto chunk = [&](const frag (&b)[U][2], frag (&nx)[U][2]) __attribute__((always_inline)) {
        const bool end = k0 + U >= p.nk;
        const Prod q = product(end ? min(st + 1, total - 1) : st);
        if (k0 == 0) {   // (ahead of the weights' loads, since loads return in order)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[0][m] = acc[1][m] = f32x4{0, 0, 0, 0};
            start();
        }
        __builtin_amdgcn_sched_barrier(0);
        load(nx, q, end ? 0 : k0 + U);   // (after the last product not used: a condition here would make every wait one for nx)
        __builtin_amdgcn_sched_barrier(0);
        const E* A = act(cur) + (HALF ? c & 7 : c) * LD + O::EPV * g + k0 * O::KS;
        if (w < p.tiles) {
            auto mma = [&](int u) __attribute__((always_inline)) {
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const frag a = *reinterpret_cast<const frag*>(A + m * 16 * LD + u * O::KS);
                    acc[0][m] = O::mma(a, b[u][0], acc[0][m]);
                    acc[1][m] = O::mma(a, b[u][1], acc[1][m]);
                }
            };
            if (k0 + U <= p.nk) {
#pragma unroll
                for (int u = 0; u < U; ++u) mma(u);   // (a second tile past the last is not used)
            } else {
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (k0 + u < p.nk) mma(u);
            }
        }
        k0 += U;
        if (end) {
            finish();
            ++st;
            k0 = 0;
            p = q;
        }
    };
    for (;;) {
        chunk(wa, wb);
        if (st == total) break;
        chunk(wb, wa);
        if (st == total) break;
    }
    asm volatile("" ::"v"(line[0]), "v"(line[1]));
    if constexpr (TRAIN) {
        for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
        if (lane == 0) red[w] = s;
        __syncthreads();
        if (tid == 0) {
            float t = 0;
            for (int i = 0; i < kRowThreads / 64; ++i) t += red[i];
            n.loss[blockIdx.x] = t * n.scale + loss0;
        }
    }
}

// workgroups for the weight gradient of a layer, columns per workgroup of a bias
// gradient (few: its loads, not its sums, take the time)
__host__ __device__ inline int dw_tiles(int N, int K, int kz) { return steps_of(N, 64) * steps_of(K, 64) * kz; }
constexpr int kColBlock = 8;

// Latency bound (1024 rows: 224 tiles of 0.5 MFLOP): the operands of eight steps,
// one split of up to 256 rows, are in flight at a time.
template <bool BF16>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void k_mlp_dw(FusedNet n, float* __restrict__ g) {
    typedef Op<BF16> O;
    typedef typename O::frag frag;
    __shared__ float sums[256 * kColBlock];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    ConstLayer& y = layer_of(n, blockIdx.y);
    int blk = blockIdx.x;
    const int tiles = dw_tiles(y.N, y.K, n.kz);
    if (blk >= tiles) {
        // bias gradient: sums of rows t, t + 256, ... and a binary tree over t
        blk -= tiles;
        if (blk >= steps_of(y.N, kColBlock)) return;
        constexpr int S = kColBlock, Q = 256 / S, J = 64 / Q;   // this thread: four rows from 4 (tid / S + Q j)
        const int q0 = tid / S, cc = tid % S, col = blk * S + cc;
        const Dev<const f32x4> src = dev<const f32x4>(y.dZ) + min(col, y.N - 1);
        f32x4 s[J];
#pragma unroll
        for (int j = 0; j < J; ++j) s[j] = f32x4{0, 0, 0, 0};
#pragma unroll 4
        for (int m = 0; m < n.ldr / 4; m += 64)   // (rows past the last are zeros)
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const int q = m + q0 + Q * j;
                if (q < n.ldr / 4) s[j] += src[(size_t)q * y.N];
            }
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) sums[(4 * (q0 + Q * j) + r) * S + cc] = s[j][r];
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            for (int e = tid; e < o * S; e += 256) sums[e] += sums[e + o * S];
            __syncthreads();
        }
        if (tid < S && col < y.N) g[y.boff + col] = sums[tid];
        return;
    }
    const int tk = steps_of(y.K, 64), z = blk % n.kz, m0 = blk / n.kz / tk * 64, k0 = blk / n.kz % tk * 64;
    const int wm = w >> 1, wn = w & 1, gq = lane >> 4, c = lane & 15;
    const int rb = z * n.klen, nk = (min(n.ldr, rb + n.klen) - rb) / O::KS, rsteps = n.ldr / O::KS;
    Dev<const frag> A[2], B[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {   // (tiles past the last repeat it: their results are not kept)
        const int m = min(m0 / 16 + wm * 2 + q, steps_of(y.N, 16) - 1), k = min(k0 / 16 + wn * 2 + q, steps_of(y.K, 16) - 1);
        A[q] = dev<const frag>(y.dT) + ((size_t)m * rsteps + rb / O::KS) * 64 + lane;
        B[q] = dev<const frag>(y.AT) + ((size_t)k * rsteps + rb / O::KS) * 64 + lane;
    }
    f32x4 acc[2][2];
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0, 0, 0, 0};
    constexpr int U = 8;
    for (int s0 = 0; s0 < nk; s0 += U) {
        frag a[U][2], b[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int s = min(s0 + u, nk - 1) * 64;
                a[u][q] = A[q][s];
                b[u][q] = B[q][s];
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u < nk)
#pragma unroll
                for (int qa = 0; qa < 2; ++qa)
#pragma unroll
                    for (int qb = 0; qb < 2; ++qb) acc[qa][qb] = O::mma(a[u][qa], b[u][qb], acc[qa][qb]);
    }
    const Dev<float> out = dev<float>(y.part) + (size_t)z * y.N * y.K;
    for (int qa = 0; qa < 2; ++qa)
        for (int qb = 0; qb < 2; ++qb)
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + wm * 32 + qa * 16 + 4 * gq + r, k = k0 + wn * 32 + qb * 16 + c;
                if (m < y.N && k < y.K) out[(size_t)m * y.K + k] = acc[qa][qb][r];
            }
}

// operand copies of weight i of layer y
template <bool BF16>
__device__ __forceinline__ void pack_weight(ConstLayer& y, unsigned i, float v) {
    typedef Op<BF16> O;
    typedef typename O::E E;
    const int nn = i / (unsigned)y.K, k = i % (unsigned)y.K;
    const E e = O::make(v);
    dev<E>(y.Wf)[frag_at<BF16>(nn, k, steps_of(y.K, O::KS))] = e;
    dev<E>(y.Wb)[frag_at<BF16>(k, nn, steps_of(y.N, O::KS))] = e;
}

// mode 0: pack the weights; 1: gradients into g; 2: and an Adam step
template <bool BF16>
__global__ __launch_bounds__(256) void k_mlp_fin(FusedNet n, int mode, float* __restrict__ p,
                                                 float* __restrict__ g, float* __restrict__ m1, float* __restrict__ m2,
                                                 float lr, float b1, float b2, float eps, float c1, float c2) {
    ConstLayer& y = layer_of(n, blockIdx.y);
    const int i = y.woff + blockIdx.x * 256 + threadIdx.x;
    if (i >= y.boff + y.N) return;
    const bool weight = i < y.boff;
    if (mode == 0) {
        if (weight) pack_weight<BF16>(y, i - y.woff, p[i]);
        return;
    }
    float gi;
    if (weight) {
        const int wsz = y.N * y.K;
        const Dev<const float> part = dev<const float>(y.part) + (i - y.woff);
        gi = 0;
        for (int z = 0; z < n.kz; ++z) gi += part[(size_t)z * wsz];
        g[i] = gi;
    } else {
        gi = g[i];
    }
    if (mode == 2) {
        adam_step(p, m1, m2, i, gi, lr, b1, b2, eps, c1, c2);
        if (weight) pack_weight<BF16>(y, i - y.woff, p[i]);
    }
}

}  // namespace
