// mlp.hip -- a small multilayer perceptron trained on the GPU: dense layers
// with GELU, mean-squared-error loss, Adam.  Used as the learned FIC
// initialiser (per-node wIE from G, wEE, wEI, SC strength, map value) and as
// the fit surrogate (per-simulation FC r and FCD KS from the parameters).  No
// counterpart in the reference.
//
// All matrix products go through one 64x64-tiled GEMM kernel on MFMA:
// BF16 operands (v_mfma_f32_16x16x32_bf16) or FP32 operands
// (v_mfma_f32_16x16x4_f32), FP32 accumulation, FP32 parameters.  Epilogues:
//   forward  Z = X W^T + b;  A = gelu(Z)          (hidden layers)
//   backward dZ_prev = (dZ W) * gelu'(Z_prev)
//   weights  dW = dZ^T X  (split over the batch, partial sums reduced in a
//            fixed order), db = column sums of dZ
// gelu(z) = z/2 (1 + erf(z/sqrt 2)).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/bnm_hip.h"
#include "pool.hpp"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

// gfx950's v_cvt_pk_bf16_f32: round to nearest even, the same bits as
// adding 0x7fff + lsb to the FP32 pattern for finite inputs
__device__ __forceinline__ unsigned short f2bf(float x) { return __builtin_bit_cast(unsigned short, (__bf16)x); }

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float z) {
    return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.3989422804014327f * expf(-0.5f * z * z);
}

constexpr int BM = 64, BN = 64, BK = 32, LDK = BK + 8;

enum Epi { EPI_STORE = 0, EPI_BIAS_GELU = 1, EPI_BIAS = 2, EPI_GELU_GRAD = 3 };

// C[M x N] (+)= op(A)[M x K] . op(B)[K x N]; element (m, k) of op(A) at
// A[m*sam + k*sak], element (k, n) of op(B) at B[k*sbk + n*sbn].  The K range
// of this workgroup is [blockIdx.z*klen, min(K, (blockIdx.z+1)*klen)); its
// output goes to C + blockIdx.z*cz.
template <bool BF16, int EPI>
__global__ __launch_bounds__(256) void k_gemm(const float* __restrict__ A, long sam, long sak,
                                              const float* __restrict__ B, long sbk, long sbn,
                                              float* __restrict__ C, long ldc, long cz, int M, int N,
                                              int K, int klen, const float* __restrict__ bias,
                                              float* __restrict__ Zout, const float* __restrict__ Zin) {
    __shared__ float As32[BF16 ? 1 : BM * LDK], Bs32[BF16 ? 1 : BN * LDK];
    __shared__ unsigned short As16[BF16 ? BM * LDK : 1], Bs16[BF16 ? BN * LDK : 1];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = w >> 1, wn = w & 1;
    const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
    const int kb = blockIdx.z * klen, ke = min(K, kb + klen);
    f32x4 acc[2][2];
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0, 0, 0, 0};
    for (int k0 = kb; k0 < ke; k0 += BK) {
        // stage a BM x BK tile of op(A) and a BN x BK tile of op(B)^T, row = m or n, col = k
        for (int e = tid; e < BM * BK; e += 256) {
            const int r = e / BK, kk = e % BK, k = k0 + kk;
            const float va = (m0 + r < M && k < ke) ? A[(long)(m0 + r) * sam + (long)k * sak] : 0.0f;
            const float vb = (n0 + r < N && k < ke) ? B[(long)k * sbk + (long)(n0 + r) * sbn] : 0.0f;
            if constexpr (BF16) {
                As16[r * LDK + kk] = f2bf(va);
                Bs16[r * LDK + kk] = f2bf(vb);
            } else {
                As32[r * LDK + kk] = va;
                Bs32[r * LDK + kk] = vb;
            }
        }
        __syncthreads();
        if constexpr (BF16) {
            u16x8 a[2], b[2];
            for (int q = 0; q < 2; ++q) {
                a[q] = *reinterpret_cast<const u16x8*>(&As16[(wm * 32 + q * 16 + (lane & 15)) * LDK + 8 * (lane >> 4)]);
                b[q] = *reinterpret_cast<const u16x8*>(&Bs16[(wn * 32 + q * 16 + (lane & 15)) * LDK + 8 * (lane >> 4)]);
            }
            for (int qa = 0; qa < 2; ++qa)
                for (int qb = 0; qb < 2; ++qb)
                    acc[qa][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, a[qa]), __builtin_bit_cast(bf16x8, b[qb]), acc[qa][qb], 0, 0, 0);
        } else {
            for (int s = 0; s < BK / 4; ++s) {
                float a[2], b[2];
                for (int q = 0; q < 2; ++q) {
                    a[q] = As32[(wm * 32 + q * 16 + (lane & 15)) * LDK + 4 * s + (lane >> 4)];
                    b[q] = Bs32[(wn * 32 + q * 16 + (lane & 15)) * LDK + 4 * s + (lane >> 4)];
                }
                for (int qa = 0; qa < 2; ++qa)
                    for (int qb = 0; qb < 2; ++qb)
                        acc[qa][qb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[qa], b[qb], acc[qa][qb], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    float* Cz = C + (long)blockIdx.z * cz;
    for (int qa = 0; qa < 2; ++qa)
        for (int qb = 0; qb < 2; ++qb)
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + wm * 32 + qa * 16 + 4 * (lane >> 4) + r;
                const int n = n0 + wn * 32 + qb * 16 + (lane & 15);
                if (m >= M || n >= N) continue;
                float v = acc[qa][qb][r];
                const long o = (long)m * ldc + n;
                if constexpr (EPI == EPI_BIAS_GELU) {
                    v += bias[n];
                    Zout[o] = v;
                    v = gelu(v);
                } else if constexpr (EPI == EPI_BIAS) {
                    v += bias[n];
                } else if constexpr (EPI == EPI_GELU_GRAD) {
                    v *= gelu_grad(Zin[o]);
                }
                Cz[o] = v;
            }
}

// out[i] = sum_z part[z*n + i], fixed order
__global__ void k_sum_parts(const float* __restrict__ part, int nz, long n, float* __restrict__ out) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        float s = 0;
        for (int z = 0; z < nz; ++z) s += part[(long)z * n + i];
        out[i] = s;
    }
}

// db[n] = sum_m dZ[m][n] (one workgroup per column block, fixed order)
__global__ void k_colsum(const float* __restrict__ dZ, int M, int N, float* __restrict__ db) {
    __shared__ float red[256];
    const int n = blockIdx.x;
    float s = 0;
    for (int m = threadIdx.x; m < M; m += blockDim.x) s += dZ[(long)m * N + n];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) db[n] = red[0];
}

// dY = 2 (Y - T) / (M*N) elementwise (gradient of the mean squared error);
// loss partial sums per workgroup
// loss_part[blockIdx.x] is overwritten, or accumulated into when `accum`
__global__ void k_mse(const float* __restrict__ Y, const float* __restrict__ T, long n, float scale,
                      float* __restrict__ dY, float* __restrict__ loss_part, int accum) {
    __shared__ float red[256];
    float s = 0;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const float d = Y[i] - T[i];
        dY[i] = 2.0f * d * scale;
        s += d * d;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss_part[blockIdx.x] = red[0] * scale + (accum ? loss_part[blockIdx.x] : 0.0f);
}

__global__ void k_fill_f32(float* __restrict__ p, int n, float v) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = v;
}

// Adam (Kingma & Ba 2015) with bias correction
__device__ __forceinline__ void adam_step(float* p, float* m1, float* m2, long i, float gi, float lr, float b1,
                                          float b2, float eps, float c1, float c2) {
    const float a = b1 * m1[i] + (1 - b1) * gi;
    const float b = b2 * m2[i] + (1 - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    p[i] -= lr * (a / c1) / (sqrtf(b / c2) + eps);
}
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m1,
                       float* __restrict__ m2, long n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        adam_step(p, m1, m2, i, g[i], lr, b1, b2, eps, c1, c2);
}

// gather rows idx[0..n) of X [*, d] into out [n, d]
__global__ void k_gather(const float* __restrict__ X, const int* __restrict__ idx, int n, int d,
                         float* __restrict__ out) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < (long)n * d; i += (long)gridDim.x * blockDim.x)
        out[i] = X[(long)idx[i / d] * d + i % d];
}

thread_local std::string g_mlp_err;
constexpr int kLossBlocks = 64;

}  // namespace

#include "mlp_fused.hpp"

struct bnm_mlp {
    int in = 0, hid = 0, depth = 0, out = 0, bf16 = 1;
    std::vector<int> dims;          // in, hid x depth, out
    std::vector<long> woff, boff;   // offsets into the flat parameter vector
    long nparam = 0;
    float *p = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;
    int cap = 0;                    // activation rows allocated
    std::vector<float*> Z, A, dZ;   // per layer [cap x dims[l+1]] (A[0] = input)
    float *part = nullptr, *loss_part = nullptr, *target = nullptr;
    long part_cap = 0;
    float *X = nullptr, *Y = nullptr, *bx = nullptr, *by = nullptr;
    int *idx = nullptr;
    int n_data = 0;
    long step = 0;
    hipStream_t st = nullptr;
    // networks of layers up to 256 wide (mlp_fused.hpp): layer pointers, the
    // weights' operand copies, and the buffers of a gradient for fcap rows
    bool fused = false;
    FusedNet net{};
    FusedLayer layer[kFusedLayers];       // net.l is their copy on the device
    void *wcopy = nullptr, *fbuf = nullptr;
    int fcap = 0, xcap = 0, loss_cap = 0, idx_cap = 0, data_cap = 0;
    float* px = nullptr;   // rows of a prediction or a loss_grad
};

namespace {

int mlp_fail(const std::string& m) {
    g_mlp_err = m;
    return BNM_E_HIP;
}

#define MCHK(expr)                                                                   \
    do {                                                                             \
        hipError_t _e = (expr);                                                      \
        if (_e != hipSuccess) return mlp_fail(std::string(#expr) + ": " + hipGetErrorString(_e)); \
    } while (0)

int ensure_rows(bnm_mlp* m, int rows) {
    if (rows <= m->cap) return BNM_OK;
    for (auto* v : {&m->Z, &m->A, &m->dZ})
        for (float*& q : *v)
            if (q) { (void)hipFree(q); q = nullptr; }
    const int L = m->depth + 1;
    m->Z.assign(L, nullptr);
    m->A.assign(L + 1, nullptr);
    m->dZ.assign(L + 1, nullptr);
    for (int l = 0; l <= L; ++l) {
        MCHK(hipMalloc(&m->A[l], (size_t)rows * m->dims[l] * sizeof(float)));
        MCHK(hipMalloc(&m->dZ[l], (size_t)rows * m->dims[l] * sizeof(float)));
    }
    for (int l = 0; l < L; ++l) MCHK(hipMalloc(&m->Z[l], (size_t)rows * m->dims[l + 1] * sizeof(float)));
    if (m->target) (void)hipFree(m->target);
    MCHK(hipMalloc(&m->target, (size_t)rows * m->out * sizeof(float)));
    m->cap = rows;
    return BNM_OK;
}

template <bool BF16, int EPI>
void gemm(bnm_mlp* m, const float* A, long sam, long sak, const float* B, long sbk, long sbn, float* C,
          long ldc, long cz, int M, int N, int K, int ksplit, const float* bias, float* Zout,
          const float* Zin) {
    int klen = (K + ksplit - 1) / ksplit;
    klen = ((klen + BK - 1) / BK) * BK;
    const int kz = (K + klen - 1) / klen;
    const dim3 grid((M + BM - 1) / BM, (N + BN - 1) / BN, kz);
    hipLaunchKernelGGL((k_gemm<BF16, EPI>), grid, dim3(256), 0, m->st, A, sam, sak, B, sbk, sbn, C, ldc,
                       cz, M, N, K, klen, bias, Zout, Zin);
}

constexpr int kChunk = 65536;   // rows of a prediction at a time

// ---- layers up to 256 wide -----------------------------------------------------
size_t padded(int n, int to) { return (size_t)((n + to - 1) / to * to); }

hipError_t put_layers(bnm_mlp* m) {
    return hipMemcpy(const_cast<FusedLayer*>(m->net.l), m->layer, m->net.L * sizeof(FusedLayer), hipMemcpyHostToDevice);
}

// Gradient buffers for `rows` rows: gelu'(Z), dZ, the operands and the
// weight gradients of the row splits.
int ensure_fused(bnm_mlp* m, int rows) {
    if (rows <= m->fcap) return BNM_OK;
    if (m->fbuf) (void)hipFree(m->fbuf);
    m->fbuf = nullptr;
    m->fcap = 0;
    const size_t es = m->bf16 ? 2 : 4, ldr = padded(rows, 32), kz = std::max(1, std::min(64, rows / 256));
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t o = off; off += (bytes + 255) / 256 * 256; return o; };
    size_t o[kFusedLayers][5];
    for (int l = 0; l < m->net.L; ++l) {
        const size_t K = m->dims[l], N = m->dims[l + 1];
        o[l][0] = take(ldr / 8 * kRowThreads * 4 * 4);
        o[l][1] = take(ldr * N * 4);
        o[l][2] = take(padded(K, 16) * ldr * es);
        o[l][3] = take(padded(N, 16) * ldr * es);
        o[l][4] = take(kz * N * K * 4);
    }
    MCHK(hipMalloc(&m->fbuf, off));
    char* b = static_cast<char*>(m->fbuf);
    for (int l = 0; l < m->net.L; ++l) {
        FusedLayer& y = m->layer[l];
        y.G = reinterpret_cast<float*>(b + o[l][0]);
        y.dZ = reinterpret_cast<float*>(b + o[l][1]);
        y.AT = b + o[l][2];
        y.dT = b + o[l][3];
        y.part = reinterpret_cast<float*>(b + o[l][4]);
    }
    MCHK(put_layers(m));
    m->fcap = rows;
    return BNM_OK;
}

int ensure_floats(float** p, int* cap, int n, size_t each) {
    if (n <= *cap) return BNM_OK;
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    *cap = 0;
    MCHK(hipMalloc(p, (size_t)n * each * sizeof(float)));
    *cap = n;
    return BNM_OK;
}

// Rows per workgroup: eight while that gives no more than one workgroup a CU (a
// step's latency counts); from two workgroups of 16 a CU on 32, so that the
// weights are read half as often from L2 (not with FP32 operands: LDS).
int block_rows(const bnm_mlp* m, int rows) { return rows <= 2048 ? 8 : m->bf16 && rows > 8192 ? 32 : 16; }

template <bool BF16, bool TRAIN>
void launch_rows(bnm_mlp* m, const FusedNet& n, int grid_rows) {
    const int R = block_rows(m, n.rows);
    const size_t smem = 2 * (size_t)R * (kFusedDim + Op<BF16>::EPV) * sizeof(typename Op<BF16>::E);
    const dim3 grid((grid_rows + R - 1) / R);
    if (R == 8) hipLaunchKernelGGL((k_mlp<BF16, 8, TRAIN>), grid, dim3(kRowThreads), smem, m->st, n);
    else if (R == 16) hipLaunchKernelGGL((k_mlp<BF16, 16, TRAIN>), grid, dim3(kRowThreads), smem, m->st, n);
    else hipLaunchKernelGGL((k_mlp<BF16, BF16 ? 32 : 16, TRAIN>), grid, dim3(kRowThreads), smem, m->st, n);
}

int fin(bnm_mlp* m, const FusedNet& n, int mode, float lr = 0, float b1 = 0, float b2 = 0, float eps = 0, float c1 = 1,
        float c2 = 1) {
    int most = 0;
    for (int l = 0; l < n.L; ++l) most = std::max(most, steps_of(m->layer[l].N * (m->layer[l].K + 1), 256));
    const dim3 grid(most, n.L);
    if (m->bf16) hipLaunchKernelGGL(k_mlp_fin<true>, grid, dim3(256), 0, m->st, n, mode, m->p, m->g, m->m1, m->m2, lr, b1, b2, eps, c1, c2);
    else hipLaunchKernelGGL(k_mlp_fin<false>, grid, dim3(256), 0, m->st, n, mode, m->p, m->g, m->m1, m->m2, lr, b1, b2, eps, c1, c2);
    MCHK(hipGetLastError());
    return BNM_OK;
}

// Many rows through a small network go layer by layer: the row blocks' workgroups cost
// the same whatever the width and come in several rounds, while a layer's product has no
// weights to wait for.  Same bits either way.  Predictions of 5 -> hidden x depth -> 1,
// row blocks / layer by layer, ms a call:
//   BF16   32 x 2:  16384 rows 0.060 / 0.065   32768 0.092 / 0.083   65536 0.166 / 0.126
//          64 x 4:                                   0.109 / 0.132         0.203 / 0.182
//         128 x 4:                                   0.121 / 0.173         0.227 / 0.260
//   FP32   32 x 2:   8192 rows 0.049 / 0.057   16384 0.069 / 0.067   65536 0.205 / 0.131
//         128 x 4:  16384 rows 0.113 / 0.143   32768 0.198 / 0.182         0.376 / 0.281
//         256 x 2:                                   0.183 / 0.193         0.348 / 0.327
//         256 x 4:                                   0.304 / 0.352         0.579 / 0.662
long weights_of(const bnm_mlp* m) {
    long w = 0;
    for (int l = 0; l <= m->depth; ++l) w += (long)m->dims[l] * m->dims[l + 1];
    return w;
}
bool predict_by_layers(const bnm_mlp* m, int rows) {
    const long w = weights_of(m), L = m->depth + 1;
    const int h = *std::max_element(m->dims.begin(), m->dims.end());
    if (m->bf16) return h <= 128 && w < 32768 && rows > 12288 + 4096 * L + 64 * h;
    return w < 131072 && rows > 8192 + 2048 * L + 64 * h + (h > 128 ? w / 4 : 0);
}
// Gradients only through one narrow hidden layer, where the derivatives that the row
// blocks keep are more than the activations of a layer (8 nodes: 131072 rows 0.63 / 0.66
// ms, 1000000 5.5 / 4.2; 64 nodes, FP32: 131072 0.79 / 0.90, 262144 1.81 / 1.64).
bool gradient_by_layers(const bnm_mlp* m, int rows) {
    const int h = *std::max_element(m->dims.begin(), m->dims.end());
    return m->depth == 1 && (m->bf16 ? h <= 32 && rows >= 327680 : h <= 64 && rows >= 229376);
}
// ... and those whose buffers are not to be had
bool gradient_fused(bnm_mlp* m, int rows) {
    if (!m->fused || gradient_by_layers(m, rows)) return false;
    if (ensure_fused(m, rows) == BNM_OK) return true;
    (void)hipGetLastError();
    return false;
}

// Partial sums of the loss that a gradient over `rows` rows leaves.
int loss_parts(const bnm_mlp* m, int rows) {
    const int R = block_rows(m, rows);
    return (int)((padded(rows, 32) + R - 1) / R);
}

// forward and back over the rows of n, and the gradient's parts
int fused_grad(bnm_mlp* m, FusedNet n) {
    n.ldr = (int)padded(n.rows, 32);
    n.scale = 1.0f / (float)((long)n.rows * m->out);
    const int ks = std::max(1, std::min(64, n.rows / 256));
    n.klen = (int)padded((n.rows + ks - 1) / ks, BK);
    n.kz = (n.rows + n.klen - 1) / n.klen;
    n.loss = m->loss_part;
    // (rows up to ldr are written too, as zeros)
    if (m->bf16) launch_rows<true, true>(m, n, n.ldr);
    else launch_rows<false, true>(m, n, n.ldr);
    int most = 0;
    for (int l = 0; l < n.L; ++l) {
        const FusedLayer& y = m->layer[l];
        most = std::max(most, dw_tiles(y.N, y.K, n.kz) + steps_of(y.N, kColBlock));
    }
    const dim3 grid(most, n.L);
    if (m->bf16) hipLaunchKernelGGL(k_mlp_dw<true>, grid, dim3(256), 0, m->st, n, m->g);
    else hipLaunchKernelGGL(k_mlp_dw<false>, grid, dim3(256), 0, m->st, n, m->g);
    m->net.kz = n.kz;
    MCHK(hipGetLastError());
    return BNM_OK;
}

// forward over `rows` rows already in A[0]; output in A[L]
int forward(bnm_mlp* m, int rows) {
    const int L = m->depth + 1;
    for (int l = 0; l < L; ++l) {
        const int K = m->dims[l], N = m->dims[l + 1];
        const float* W = m->p + m->woff[l];
        const float* b = m->p + m->boff[l];
        const bool last = l == L - 1;
        if (m->bf16) {
            if (last) gemm<true, EPI_BIAS>(m, m->A[l], K, 1, W, 1, K, m->A[l + 1], N, 0, rows, N, K, 1, b, nullptr, nullptr);
            else gemm<true, EPI_BIAS_GELU>(m, m->A[l], K, 1, W, 1, K, m->A[l + 1], N, 0, rows, N, K, 1, b, m->Z[l], nullptr);
        } else {
            if (last) gemm<false, EPI_BIAS>(m, m->A[l], K, 1, W, 1, K, m->A[l + 1], N, 0, rows, N, K, 1, b, nullptr, nullptr);
            else gemm<false, EPI_BIAS_GELU>(m, m->A[l], K, 1, W, 1, K, m->A[l + 1], N, 0, rows, N, K, 1, b, m->Z[l], nullptr);
        }
    }
    MCHK(hipGetLastError());
    return BNM_OK;
}

// gradient into m->g for `rows` rows with targets in m->target; the loss goes
// to m->loss_part (kLossBlocks partial sums, added to what is there when
// `accum`), and to *loss when given (synchronises)
int backward(bnm_mlp* m, int rows, float* loss, int accum = 0) {
    const int L = m->depth + 1;
    const long nout = (long)rows * m->out;
    const int lb = kLossBlocks;
    hipLaunchKernelGGL(k_mse, dim3(lb), dim3(256), 0, m->st, m->A[L], m->target, nout, 1.0f / (float)nout,
                       m->dZ[L], m->loss_part, accum);
    for (int l = L - 1; l >= 0; --l) {
        const int K = m->dims[l], N = m->dims[l + 1];
        const float* W = m->p + m->woff[l];
        // dW[N x K] = dZ_{l+1}^T [N x rows] . A_l [rows x K], split over rows
        const int ks = std::max(1, std::min(64, rows / 256));
        const long wsz = (long)N * K;
        if (m->part_cap < wsz * ks) {
            if (m->part) (void)hipFree(m->part);
            MCHK(hipMalloc(&m->part, (size_t)wsz * ks * sizeof(float)));
            m->part_cap = wsz * ks;
        }
        if (m->bf16)
            gemm<true, EPI_STORE>(m, m->dZ[l + 1], 1, N, m->A[l], K, 1, m->part, K, wsz, N, K, rows, ks, nullptr, nullptr, nullptr);
        else
            gemm<false, EPI_STORE>(m, m->dZ[l + 1], 1, N, m->A[l], K, 1, m->part, K, wsz, N, K, rows, ks, nullptr, nullptr, nullptr);
        int klen = (rows + ks - 1) / ks;
        klen = ((klen + BK - 1) / BK) * BK;
        const int kz = (rows + klen - 1) / klen;
        hipLaunchKernelGGL(k_sum_parts, dim3(256), dim3(256), 0, m->st, m->part, kz, wsz, m->g + m->woff[l]);
        hipLaunchKernelGGL(k_colsum, dim3(N), dim3(256), 0, m->st, m->dZ[l + 1], rows, N, m->g + m->boff[l]);
        if (l > 0) {
            // dZ_l = (dZ_{l+1} . W) * gelu'(Z_{l-1})
            if (m->bf16)
                gemm<true, EPI_GELU_GRAD>(m, m->dZ[l + 1], N, 1, W, K, 1, m->dZ[l], K, 0, rows, K, N, 1, nullptr, nullptr, m->Z[l - 1]);
            else
                gemm<false, EPI_GELU_GRAD>(m, m->dZ[l + 1], N, 1, W, K, 1, m->dZ[l], K, 0, rows, K, N, 1, nullptr, nullptr, m->Z[l - 1]);
        }
    }
    MCHK(hipGetLastError());
    if (loss) {
        std::vector<float> lp(lb);
        MCHK(hipMemcpyAsync(lp.data(), m->loss_part, lb * sizeof(float), hipMemcpyDeviceToHost, m->st));
        MCHK(hipStreamSynchronize(m->st));
        double s = 0;
        for (float v : lp) s += v;
        *loss = (float)s;
    }
    return BNM_OK;
}

}  // namespace

extern "C" {

const char* bnm_mlp_last_error(void) { return g_mlp_err.c_str(); }

bnm_mlp* bnm_mlp_create(int in_dim, int hidden, int depth, int out_dim, int bf16, unsigned seed,
                        int* status) {
    auto set = [&](int s) { if (status) *status = s; };
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
        g_mlp_err = "no HIP device";
        set(BNM_E_NODEV);
        return nullptr;
    }
    if (in_dim < 1 || hidden < 1 || depth < 1 || out_dim < 1) {
        g_mlp_err = "bad MLP shape";
        set(BNM_E_ARG);
        return nullptr;
    }
    auto* m = new bnm_mlp;
    m->loss_cap = kLossBlocks;
    m->in = in_dim; m->hid = hidden; m->depth = depth; m->out = out_dim; m->bf16 = bf16 != 0;
    m->dims.push_back(in_dim);
    for (int i = 0; i < depth; ++i) m->dims.push_back(hidden);
    m->dims.push_back(out_dim);
    long off = 0;
    for (int l = 0; l <= depth; ++l) {
        m->woff.push_back(off);
        off += (long)m->dims[l] * m->dims[l + 1];
        m->boff.push_back(off);
        off += m->dims[l + 1];
    }
    m->nparam = off;
    // He-style uniform init in [-sqrt(6/fan_in), sqrt(6/fan_in)] (weights), zero biases
    std::vector<float> h(off, 0.0f);
    std::mt19937 gen(seed);
    for (int l = 0; l <= depth; ++l) {
        const float a = std::sqrt(6.0f / m->dims[l]) * (l == depth ? 0.5f : 1.0f);
        std::uniform_real_distribution<float> u(-a, a);
        for (long i = 0; i < (long)m->dims[l] * m->dims[l + 1]; ++i) h[m->woff[l] + i] = u(gen);
    }
    bool ok = hipStreamCreateWithFlags(&m->st, hipStreamNonBlocking) == hipSuccess &&
              hipMalloc(&m->p, off * sizeof(float)) == hipSuccess &&
              hipMalloc(&m->g, off * sizeof(float)) == hipSuccess &&
              hipMalloc(&m->m1, off * sizeof(float)) == hipSuccess &&
              hipMalloc(&m->m2, off * sizeof(float)) == hipSuccess &&
              hipMalloc(&m->loss_part, kLossBlocks * sizeof(float)) == hipSuccess &&
              hipMemcpy(m->p, h.data(), off * sizeof(float), hipMemcpyHostToDevice) == hipSuccess &&
              hipMemset(m->m1, 0, off * sizeof(float)) == hipSuccess &&
              hipMemset(m->m2, 0, off * sizeof(float)) == hipSuccess;
    if (!ok) {
        g_mlp_err = "MLP allocation failed";
        set(BNM_E_HIP);
        bnm_mlp_destroy(m);
        return nullptr;
    }
    m->fused = depth + 1 <= kFusedLayers && std::max({in_dim, hidden, out_dim}) <= kFusedDim;
    if (m->fused) {
        const size_t es = m->bf16 ? 2 : 4;
        const int ks = m->bf16 ? 32 : 16;
        m->net.L = depth + 1;
        size_t off = 0, of[kFusedLayers], ob[kFusedLayers];
        for (int l = 0; l <= depth; ++l) {
            const int K = m->dims[l], N = m->dims[l + 1];
            of[l] = off;
            off += padded(N, 16) * padded(K, ks) * es;
            ob[l] = off;
            off += padded(K, 16) * padded(N, ks) * es;
        }
        off = (off + 255) / 256 * 256;
        ok = hipMalloc(&m->wcopy, off + sizeof(m->layer)) == hipSuccess && hipMemset(m->wcopy, 0, off) == hipSuccess &&
             hipDeviceSynchronize() == hipSuccess;
        m->net.W = static_cast<const unsigned*>(m->wcopy);
        m->net.wwords = (unsigned)(off / 4);
        m->net.l = reinterpret_cast<FusedLayer*>(static_cast<char*>(m->wcopy) + off);
        for (int l = 0; l <= depth && ok; ++l) {
            FusedLayer& y = m->layer[l] = FusedLayer{};
            y.K = m->dims[l];
            y.N = m->dims[l + 1];
            y.Wf = static_cast<char*>(m->wcopy) + of[l];
            y.Wb = static_cast<char*>(m->wcopy) + ob[l];
            y.b = m->p + m->boff[l];
            y.woff = (int)m->woff[l];
            y.boff = (int)m->boff[l];
        }
        if (!ok || put_layers(m) != hipSuccess || fin(m, m->net, 0) != BNM_OK) {
            g_mlp_err = "MLP allocation failed";
            set(BNM_E_HIP);
            bnm_mlp_destroy(m);
            return nullptr;
        }
    }
    set(BNM_OK);
    return m;
}

void bnm_mlp_destroy(bnm_mlp* m) {
    if (!m) return;
    for (float* q : {m->p, m->g, m->m1, m->m2, m->part, m->loss_part, m->target, m->X, m->Y, m->bx, m->by})
        if (q) (void)hipFree(q);
    if (m->idx) (void)hipFree(m->idx);
    for (void* q : {m->wcopy, m->fbuf, (void*)m->px})
        if (q) (void)hipFree(q);
    for (auto* v : {&m->Z, &m->A, &m->dZ})
        for (float* q : *v)
            if (q) (void)hipFree(q);
    if (m->st) (void)hipStreamDestroy(m->st);
    delete m;
}

long bnm_mlp_num_params(bnm_mlp* m) { return m ? m->nparam : -1; }

int bnm_mlp_get_params(bnm_mlp* m, float* out) {
    if (!m || !out) return BNM_E_ARG;
    MCHK(hipStreamSynchronize(m->st));
    MCHK(hipMemcpy(out, m->p, m->nparam * sizeof(float), hipMemcpyDeviceToHost));
    return BNM_OK;
}

int bnm_mlp_set_params(bnm_mlp* m, const float* in) {
    if (!m || !in) return BNM_E_ARG;
    MCHK(hipStreamSynchronize(m->st));
    MCHK(hipMemcpy(m->p, in, m->nparam * sizeof(float), hipMemcpyHostToDevice));
    return m->fused ? fin(m, m->net, 0) : BNM_OK;
}

// Y[n x out] = f(X[n x in])
int bnm_mlp_predict(bnm_mlp* m, const float* X, int n, float* Y) {
    if (!m || !X || !Y || n < 1) return BNM_E_ARG;
    const int chunk = kChunk;
    if (m->fused && !predict_by_layers(m, std::min(n, chunk))) {
        int e = ensure_floats(&m->px, &m->xcap, std::min(n, chunk), m->in + m->out);
        if (e) return e;
        FusedNet f = m->net;
        f.X = m->px;
        f.Y = m->px + (size_t)m->xcap * m->in;
        for (int s = 0; s < n; s += chunk) {
            f.rows = std::min(chunk, n - s);
            MCHK(hipMemcpyAsync(m->px, X + (long)s * m->in, (size_t)f.rows * m->in * sizeof(float), hipMemcpyHostToDevice, m->st));
            if (m->bf16) launch_rows<true, false>(m, f, f.rows);
            else launch_rows<false, false>(m, f, f.rows);
            MCHK(hipGetLastError());
            MCHK(hipMemcpyAsync(Y + (long)s * m->out, f.Y, (size_t)f.rows * m->out * sizeof(float), hipMemcpyDeviceToHost, m->st));
            MCHK(hipStreamSynchronize(m->st));
        }
        return BNM_OK;
    }
    for (int s = 0; s < n; s += chunk) {
        const int r = std::min(chunk, n - s);
        int e = ensure_rows(m, r);
        if (e) return e;
        MCHK(hipMemcpyAsync(m->A[0], X + (long)s * m->in, (size_t)r * m->in * sizeof(float), hipMemcpyHostToDevice, m->st));
        if ((e = forward(m, r))) return e;
        MCHK(hipMemcpyAsync(Y + (long)s * m->out, m->A[m->depth + 1], (size_t)r * m->out * sizeof(float),
                            hipMemcpyDeviceToHost, m->st));
        MCHK(hipStreamSynchronize(m->st));
    }
    return BNM_OK;
}

// Loss (mean squared error over n x out) and its gradient w.r.t. the flat
// parameter vector at the current parameters.
int bnm_mlp_loss_grad(bnm_mlp* m, const float* X, const float* T, int n, float* loss, float* grad) {
    if (!m || !X || !T || n < 1) return BNM_E_ARG;
    int e = 0;
    if (gradient_fused(m, n)) {
        const int parts = loss_parts(m, n);
        if ((e = ensure_floats(&m->px, &m->xcap, n, m->in + m->out))) return e;
        if ((e = ensure_floats(&m->loss_part, &m->loss_cap, parts, 1))) return e;
        FusedNet f = m->net;
        f.rows = n;
        f.X = m->px;
        f.T = m->px + (size_t)m->xcap * m->in;
        MCHK(hipMemcpyAsync(m->px, X, (size_t)n * m->in * sizeof(float), hipMemcpyHostToDevice, m->st));
        MCHK(hipMemcpyAsync(const_cast<float*>(f.T), T, (size_t)n * m->out * sizeof(float), hipMemcpyHostToDevice, m->st));
        if ((e = fused_grad(m, f))) return e;
        if ((e = fin(m, m->net, 1))) return e;
        std::vector<float> lp(parts);
        MCHK(hipMemcpyAsync(lp.data(), m->loss_part, parts * sizeof(float), hipMemcpyDeviceToHost, m->st));
        if (grad) MCHK(hipMemcpyAsync(grad, m->g, m->nparam * sizeof(float), hipMemcpyDeviceToHost, m->st));
        MCHK(hipStreamSynchronize(m->st));
        if (loss) {
            double s = 0;
            for (float v : lp) s += v;
            *loss = (float)s;
        }
        return BNM_OK;
    }
    if ((e = ensure_rows(m, n))) return e;
    MCHK(hipMemcpyAsync(m->A[0], X, (size_t)n * m->in * sizeof(float), hipMemcpyHostToDevice, m->st));
    MCHK(hipMemcpyAsync(m->target, T, (size_t)n * m->out * sizeof(float), hipMemcpyHostToDevice, m->st));
    if ((e = forward(m, n))) return e;
    if ((e = backward(m, n, loss))) return e;
    if (grad) MCHK(hipMemcpy(grad, m->g, m->nparam * sizeof(float), hipMemcpyDeviceToHost));
    MCHK(hipStreamSynchronize(m->st));
    return BNM_OK;
}

// Uploads a training set (X [n x in], T [n x out]) to the device.
int bnm_mlp_set_data(bnm_mlp* m, const float* X, const float* T, int n) {
    if (!m || !X || !T || n < 1) return BNM_E_ARG;
    MCHK(hipStreamSynchronize(m->st));
    if (n > m->data_cap) {   // (a set that fits goes where the last one was)
        for (float** q : {&m->X, &m->Y})
            if (*q) { (void)hipFree(*q); *q = nullptr; }
        m->n_data = m->data_cap = 0;
        MCHK(hipMalloc(&m->X, (size_t)n * m->in * sizeof(float)));
        MCHK(hipMalloc(&m->Y, (size_t)n * m->out * sizeof(float)));
        m->data_cap = n;
    }
    MCHK(hipMemcpy(m->X, X, (size_t)n * m->in * sizeof(float), hipMemcpyHostToDevice));
    MCHK(hipMemcpy(m->Y, T, (size_t)n * m->out * sizeof(float), hipMemcpyHostToDevice));
    m->n_data = n;
    return BNM_OK;
}

// Adam on shuffled mini-batches of the uploaded set; loss[e] = mean batch loss
// of epoch e.
int bnm_mlp_train(bnm_mlp* m, int epochs, int batch, float lr, unsigned seed, float* loss) {
    if (!m || m->n_data < 1 || batch < 1 || epochs < 1) return BNM_E_ARG;
    batch = std::min(batch, m->n_data);
    const bool fused = gradient_fused(m, batch);
    int e = fused ? BNM_OK : ensure_rows(m, batch);
    if (e) return e;
    const int parts = fused ? loss_parts(m, batch) : kLossBlocks;
    if ((e = ensure_floats(&m->loss_part, &m->loss_cap, parts, 1))) return e;
    if (m->idx_cap < m->n_data) {
        if (m->idx) { (void)hipFree(m->idx); m->idx = nullptr; }
        m->idx_cap = 0;
        MCHK(hipMalloc(&m->idx, (size_t)m->n_data * sizeof(int)));
        m->idx_cap = m->n_data;
    }
    std::mt19937 gen(seed);
    std::vector<int> perm(m->n_data);
    for (int i = 0; i < m->n_data; ++i) perm[i] = i;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const int nb = m->n_data / batch;
    std::vector<float> lp(parts);
    for (int ep = 0; ep < epochs; ++ep) {
        std::shuffle(perm.begin(), perm.end(), gen);
        // the previous epoch's kernels read m->idx: the synchronous copy waits for them
        MCHK(hipStreamSynchronize(m->st));
        MCHK(hipMemcpy(m->idx, perm.data(), (size_t)m->n_data * sizeof(int), hipMemcpyHostToDevice));
        hipLaunchKernelGGL(k_fill_f32, dim3(1), dim3(64), 0, m->st, m->loss_part, parts, 0.0f);
        for (int b = 0; b < nb; ++b) {
            const int* ib = m->idx + (long)b * batch;
            if (fused) {
                FusedNet f = m->net;
                f.rows = batch;
                f.X = m->X;
                f.T = m->Y;
                f.idx = ib;
                f.accum = 1;
                if ((e = fused_grad(m, f))) return e;
                ++m->step;
                const float c1 = 1 - std::pow(b1, (float)m->step), c2 = 1 - std::pow(b2, (float)m->step);
                if ((e = fin(m, m->net, 2, lr, b1, b2, eps, c1, c2))) return e;
                continue;
            }
            hipLaunchKernelGGL(k_gather, dim3(256), dim3(256), 0, m->st, m->X, ib, batch, m->in, m->A[0]);
            hipLaunchKernelGGL(k_gather, dim3(256), dim3(256), 0, m->st, m->Y, ib, batch, m->out, m->target);
            if ((e = forward(m, batch))) return e;
            if ((e = backward(m, batch, nullptr, 1))) return e;
            ++m->step;
            const float c1 = 1 - std::pow(b1, (float)m->step), c2 = 1 - std::pow(b2, (float)m->step);
            hipLaunchKernelGGL(k_adam, dim3(256), dim3(256), 0, m->st, m->p, m->g, m->m1, m->m2, m->nparam, lr, b1,
                               b2, eps, c1, c2);
        }
        MCHK(hipGetLastError());
        // the row blocks' copies of the weights
        if (m->fused && !fused && (e = fin(m, m->net, 0))) return e;
        if (loss) {
            MCHK(hipMemcpyAsync(lp.data(), m->loss_part, parts * sizeof(float), hipMemcpyDeviceToHost, m->st));
            MCHK(hipStreamSynchronize(m->st));
            double ls = 0;
            for (float v : lp) ls += v;
            loss[ep] = (float)(ls / nb);
        }
    }
    MCHK(hipStreamSynchronize(m->st));
    return BNM_OK;
}

}  // extern "C"
