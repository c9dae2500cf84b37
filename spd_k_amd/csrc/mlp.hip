// Per-element MLP for the Picard initial guess: BF16 MFMA forward and
// backward kernels with FP32 accumulation, and Adam with FP32 master weights.
//
// Network: x (din) -> GELU(W1 x + b1) -> GELU(W2 h1 + b2) -> W3 h2 + b3 (dout),
// GELU(z) = z/2 (1 + erf(z / sqrt 2)). Weights are stored "out x in"
// (row n holds the weights of output n); every feature dimension is padded
// to a multiple of 64 with zero weights.
//
// Two GEMM kernels on v_mfma_f32_16x16x32_bf16, C(m, n) = sum_k A(m, k) B(k, n):
// k_gemm where both operands are contiguous along k (forward, input gradients)
// and k_gemm_wgrad where both are contiguous along their output index (weight
// gradients: k is the batch row).
// Lane layout of that instruction (checked against a CPU product): lane l
// holds A[l%16][8(l/16)+j], B[8(l/16)+j][l%16] (j < 8) and C[4(l/16)+i][l%16]
// (i < 4).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>
#include "ctx.hpp"

using namespace spdk;

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

struct spdk_mlp {
    int dims[4] = {};  // padded: in, h1, h2, out
    int din = 0, dout = 0;
    int cap = 0;       // batch capacity of the activation buffers
    hipStream_t stream = nullptr;
    long nparam = 0;                          // padded parameters
    float *par = nullptr, *mom = nullptr, *var = nullptr;  // W1, b1, W2, b2, W3, b3 and their Adam moments
    float* grad = nullptr;                    // gradients in the same order, then the loss
    float *W[3] = {}, *b[3] = {};             // FP32 master parameters (in par)
    bf16 *Wb[3] = {}, *WbT[3] = {};           // BF16 copies, out x in and in x out
    float *gW[3] = {}, *gb[3] = {};           // gradients (in grad)
    bf16* X = nullptr;                        // (cap, d0)
    float* Z[3] = {};                         // pre-activations (cap, d_{l+1})
    bf16* H[2] = {};                          // activations (cap, d1), (cap, d2)
    bf16 *dZb[2] = {};                        // BF16 copies of layer gradients (ping-pong)
    float* loss = nullptr;                    // device scalar (in grad)
    long long step = 0;
    std::vector<void*> owned;
};

namespace {

enum { EPI_BIAS_GELU = 0, EPI_BIAS = 1, EPI_GELU_BWD = 2 };

// C(m, n) = sum_k A[m * lda + k] B[n * ldb + k]; N and K multiples of 64 (the
// padded layer sizes), lda and ldb multiples of 8.
struct GemmP {
    const bf16* A;
    long lda;
    const bf16* B;
    long ldb;
    int M, N, K;
    const float* bias;
    float* C;         // pre-activation (null: not stored)
    long ldc;
    int ncol;         // columns of C that are stored
    bf16* Cb;
    long ldcb;
    const float* Zp;  // pre-activation for the GELU derivative
    long ldz;
    float* colsum;    // EPI_GELU_BWD: column sums added here (bias gradient)
};

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_d(float z) {
    return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

constexpr int TK = 64, LDK = TK + 8;  // LDS rows padded to 144 bytes

// One workgroup: a BT x BT output tile, its four waves a 2 x 2 arrangement of
// (BT/2) x (BT/2) each, K in steps of 64; the next step's rows are loaded
// into registers while the MFMAs of the current one run. BT = 128 reads each
// operand half as often and is taken where its tiles still fill the chip
// (>= 512 workgroups, two per CU); the training batches (4096 rows by 256)
// have 64 such tiles, so they keep BT = 64.
template <int BT, int EPI>
__global__ void __launch_bounds__(256) k_gemm(GemmP p) {
    constexpr int R = BT / 32;  // 16-wide fragments per wave and side
    constexpr int NL = BT / 32;  // 16-byte loads per thread and operand
    __shared__ __align__(16) bf16 As[BT * LDK];
    __shared__ __align__(16) bf16 Bs[BT * LDK];
    const int tid = threadIdx.x, w = tid / 64, l = tid % 64;
    const int m0 = blockIdx.y * BT, n0 = blockIdx.x * BT;
    const int wm = (w / 2) * (BT / 2), wn = (w % 2) * (BT / 2);
    const int lr = tid / 8, lk = (tid % 8) * 8;  // staging: rows lr + 32 i, 8 values from k offset lk
    floatx4 acc[R][R];
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
        for (int j = 0; j < R; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    bf16x8 ra[NL], rb[NL];
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            // rows and columns past the end are clamped: they only reach outputs that are not stored
            const int m = min(m0 + lr + 32 * i, p.M - 1), n = min(n0 + lr + 32 * i, p.N - 1);
            ra[i] = *(const bf16x8*)(p.A + (long)m * p.lda + k0 + lk);
            rb[i] = *(const bf16x8*)(p.B + (long)n * p.ldb + k0 + lk);
        }
    };
    load(0);
    for (int k0 = 0; k0 < p.K; k0 += TK) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NL; i++) {
            *(bf16x8*)(As + (lr + 32 * i) * LDK + lk) = ra[i];
            *(bf16x8*)(Bs + (lr + 32 * i) * LDK + lk) = rb[i];
        }
        __syncthreads();
        if (k0 + TK < p.K) load(k0 + TK);
#pragma unroll
        for (int kk = 0; kk < TK; kk += 32) {
            bf16x8 fa[R], fb[R];
#pragma unroll
            for (int i = 0; i < R; i++) {
                fa[i] = *(const bf16x8*)(As + (wm + 16 * i + l % 16) * LDK + kk + 8 * (l / 16));
                fb[i] = *(const bf16x8*)(Bs + (wn + 16 * i + l % 16) * LDK + kk + 8 * (l / 16));
            }
#pragma unroll
            for (int i = 0; i < R; i++)
#pragma unroll
                for (int j = 0; j < R; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
    }
    // epilogue: lane l holds C[wm + 16 i + 4 (l/16) + r][wn + 16 j + l%16]
#pragma unroll
    for (int j = 0; j < R; j++) {
        const int n = n0 + wn + 16 * j + l % 16;
        const bool in = n < p.N;
        const float bias = EPI != EPI_GELU_BWD && in ? p.bias[n] : 0.f;
        float cs = 0.f;
#pragma unroll
        for (int i = 0; i < R; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + wm + 16 * i + 4 * (l / 16) + r;
                if (m >= p.M || !in) continue;
                float v = acc[i][j][r];
                if (EPI == EPI_GELU_BWD) {
                    v *= gelu_d(p.Zp[(long)m * p.ldz + n]);
                    cs += v;
                    p.Cb[(long)m * p.ldcb + n] = (bf16)v;
                } else {
                    v += bias;
                    if (p.C && n < p.ncol) p.C[(long)m * p.ldc + n] = v;
                    if (EPI == EPI_BIAS_GELU) p.Cb[(long)m * p.ldcb + n] = (bf16)gelu(v);
                }
            }
        if (EPI == EPI_GELU_BWD) {  // the wave's rows of column n, then one atomic per column and wave
            cs += __shfl_xor(cs, 16);
            cs += __shfl_xor(cs, 32);
            if (l < 16 && in) atomicAdd(&p.colsum[n], cs);
        }
    }
}

// Weight gradient gW[n][k] += sum_m dZ[m][n] X[m][k] over the batch rows
// [z * chunk, (z + 1) * chunk) of workgroup z: 64 x 64 outputs, rows in steps
// of 64. Both operands are contiguous along their output index, so a thread
// loads 8 columns of two adjacent rows (16-byte loads, whole lines per 8
// lanes) and writes them to LDS as (m, m+1) pairs, row n holding the m of its
// column; the 16-byte chunks of a row are permuted by (n / 8) % 8 so that the
// eight column groups a wave writes fall in different banks. (Reading the
// operands element by element along m, two bytes at a time, took 25 us per
// product at 4096 rows, 1280 x 256.)
struct WgradP {
    const bf16* dZ;
    const bf16* X;
    int N, K;  // outputs (multiples of 64)
    int rows, chunk;
    float* gW;
};
__global__ void __launch_bounds__(256) k_gemm_wgrad(WgradP p) {
    __shared__ __align__(16) bf16 As[64 * LDK];
    __shared__ __align__(16) bf16 Bs[64 * LDK];
    const int tid = threadIdx.x, w = tid / 64, l = tid % 64;
    const int n0 = blockIdx.y * 64, k0 = blockIdx.x * 64;
    const int mb = blockIdx.z * p.chunk, me = min(p.rows, mb + p.chunk);
    const int wm = (w / 2) * 32, wn = (w % 2) * 32;
    const int cg = tid % 8, pair = tid / 8;  // 8 columns from 8 cg, rows 2 pair and 2 pair + 1
    floatx4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    bf16x8 a0, a1, b0, b1;
    const bf16x8 zero = {};
    auto load = [&](int m) {
        const int r = m + 2 * pair;
        a0 = r < me ? *(const bf16x8*)(p.dZ + (long)r * p.N + n0 + 8 * cg) : zero;
        a1 = r + 1 < me ? *(const bf16x8*)(p.dZ + (long)(r + 1) * p.N + n0 + 8 * cg) : zero;
        b0 = r < me ? *(const bf16x8*)(p.X + (long)r * p.K + k0 + 8 * cg) : zero;
        b1 = r + 1 < me ? *(const bf16x8*)(p.X + (long)(r + 1) * p.K + k0 + 8 * cg) : zero;
    };
    typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));
    // element offset of row n, values m = 8 c .. 8 c + 7
    auto at = [](int n, int c) { return n * LDK + ((c ^ (n / 8)) % 8) * 8; };
    load(mb);
    for (int m = mb; m < me; m += TK) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int o = at(8 * cg + j, pair / 4) + 2 * (pair % 4);
            *(bf16x2*)(As + o) = bf16x2{a0[j], a1[j]};
            *(bf16x2*)(Bs + o) = bf16x2{b0[j], b1[j]};
        }
        __syncthreads();
        if (m + TK < me) load(m + TK);
#pragma unroll
        for (int kk = 0; kk < TK; kk += 32) {
            bf16x8 fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                fa[i] = *(const bf16x8*)(As + at(wm + 16 * i + l % 16, kk / 8 + l / 16));
                fb[i] = *(const bf16x8*)(Bs + at(wn + 16 * i + l % 16, kk / 8 + l / 16));
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                atomicAdd(&p.gW[(long)(n0 + wm + 16 * i + 4 * (l / 16) + r) * p.K + k0 + wn + 16 * j + l % 16], acc[i][j][r]);
}

// loss = mean (Y - T)^2 over the first dout columns; dYb = 2 (Y - T) / count
// in BF16 (padded columns get zero gradient), the FP32 column sums of it (the
// bias gradient) added to gb. A thread owns one column and kMseRows rows, so a
// column's sum and the workgroup's loss cost one atomic each (one atomic on
// the loss per 256 values, from 20,480 workgroups, took 263 us at 4096 x 1280).
// The atomics add in any order: bias gradients, like the weights', differ from
// run to run in their last bits.
constexpr int kMseRows = 32;
__global__ void __launch_bounds__(256) k_mse(const float* Y, long ldy, const float* T, long ldt, int M, int dout,
                                             int dpad, float inv_count, bf16* dYb, float* gb, float* loss) {
    const int n = blockIdx.x * 256 + threadIdx.x, m0 = blockIdx.y * kMseRows, m1 = min(M, m0 + kMseRows);
    float acc = 0.f, cs = 0.f;
    if (n < dpad) {
#pragma unroll 8
        for (int m = m0; m < m1; m++) {
            float g = 0.f;
            if (n < dout) {
                const float d = Y[(long)m * ldy + n] - T[(long)m * ldt + n];
                acc += d * d;
                g = 2.f * d * inv_count;
            }
            cs += g;
            dYb[(long)m * dpad + n] = (bf16)g;
        }
        atomicAdd(&gb[n], cs);
    }
    __shared__ float red[4];
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) acc += __shfl_xor(acc, s);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = acc;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(loss, (red[0] + red[1] + red[2] + red[3]) * inv_count);
}

__global__ void k_fill(float* p, long n, float v) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

// Adam (bias-corrected) on the FP32 masters of every layer in one launch
// (parameters, moments and gradients are each one array in the order W1, b1,
// W2, b2, W3, b3); refreshes the BF16 copies of the weight matrices in both
// layouts (rows x cols = out x in).
struct AdamP {
    float *w, *m, *v;
    const float* g;
    long end[6];  // end of each part
    int rows[3], cols[3];
    bf16 *wb[3], *wbT[3];
    float lr, b1, b2, eps, c1, c2;
};
__global__ void k_adam(AdamP p) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < p.end[5]; i += (long)gridDim.x * blockDim.x) {
        const float gi = p.g[i];
        const float mi = p.b1 * p.m[i] + (1.f - p.b1) * gi;
        const float vi = p.b2 * p.v[i] + (1.f - p.b2) * gi * gi;
        p.m[i] = mi;
        p.v[i] = vi;
        const float wi = p.w[i] - p.lr * (mi * p.c1) / (sqrtf(vi * p.c2) + p.eps);
        p.w[i] = wi;
#pragma unroll
        for (int l = 0; l < 3; l++) {
            const long o = i - (l ? p.end[2 * l - 1] : 0);
            if (o >= 0 && i < p.end[2 * l]) {
                p.wb[l][o] = (bf16)wi;
                const long r = o / p.cols[l], c = o % p.cols[l];
                p.wbT[l][c * p.rows[l] + r] = (bf16)wi;
            }
        }
    }
}

__global__ void k_to_bf16(const float* src, bf16* dst, bf16* dstT, long n, int cols, int rows) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        dst[i] = (bf16)src[i];
        if (dstT) dstT[(i % cols) * rows + i / cols] = (bf16)src[i];
    }
}

// FP32 rows (M x din, leading dimension ld) into the padded BF16 input.
__global__ void k_pack_input(const float* Xf, long ld, int M, int din, int dpad, bf16* X) {
    const long total = (long)M * dpad;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        const int m = (int)(i / dpad), n = (int)(i % dpad);
        X[i] = (bf16)(n < din ? Xf[(long)m * ld + n] : 0.0f);
    }
}

// dst[r][:] = src[idx[r]][:] for r < n (cols values per row)
__global__ void k_gather(const float* src, long ld, const int* idx, int n, int cols, float* dst) {
    const long total = (long)n * cols;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        const int r = (int)(i / cols), c = (int)(i % cols);
        dst[i] = src[(long)idx[r] * ld + c];
    }
}

// flags[r] = 1 if every value of row r is finite with magnitude < maxabs
__global__ void k_rows_ok(const float* Y, long ld, int rows, int cols, float maxabs, unsigned char* flags) {
    const int r = blockIdx.x;
    if (r >= rows) return;
    __shared__ int bad;
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
    for (int c = threadIdx.x; c < cols; c += blockDim.x) {
        const float v = Y[(long)r * ld + c];
        if (!(fabsf(v) < maxabs)) bad = 1;
    }
    __syncthreads();
    if (threadIdx.x == 0) flags[r] = bad ? 0 : 1;
}

inline unsigned nb(long n, int bs) { long b = (n + bs - 1) / bs; return (unsigned)(b > 65535 * 4 ? 65535 * 4 : b); }

template <int EPI>
int gemm(hipStream_t st, const GemmP& p) {
    const long big = (long)((p.N + 127) / 128) * ((p.M + 127) / 128);
    const int bt = big >= 512 ? 128 : 64;
    const dim3 grid((p.N + bt - 1) / bt, (p.M + bt - 1) / bt);
    if (grid.y > 65535 * 16) { set_error("mlp: batch too large for one launch"); return SPDK_E_ARG; }
    if (bt == 128) hipLaunchKernelGGL((k_gemm<128, EPI>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((k_gemm<64, EPI>), grid, dim3(256), 0, st, p);
    SPDK_LAUNCH_CHECK("k_gemm");
    return SPDK_OK;
}

int alloc(spdk_mlp* net, void** p, size_t bytes) {
    SPDK_CHECK(hipMalloc(p, bytes));
    net->owned.push_back(*p);
    SPDK_CHECK(hipMemsetAsync(*p, 0, bytes, net->stream));
    return SPDK_OK;
}

// forward over B rows already packed in net->X. Training (Y null): the
// pre-activations of every layer stay in net->Z. Inference: only the outputs
// are kept, written to Y (B x dout, leading dimension ldy).
int forward(spdk_mlp* net, int B, float* Y = nullptr, long ldy = 0) {
    const int* d = net->dims;
    const bf16* in = net->X;
    for (int l = 0; l < 3; l++) {
        GemmP p{};
        p.A = in;
        p.lda = d[l];
        p.B = net->Wb[l];  // B(k, n) = W[n][k]
        p.ldb = d[l];
        p.M = B;
        p.N = d[l + 1];
        p.K = d[l];
        p.bias = net->b[l];
        p.C = Y ? (l < 2 ? nullptr : Y) : net->Z[l];
        p.ldc = Y ? ldy : d[l + 1];
        p.ncol = Y ? net->dout : d[l + 1];
        p.Cb = l < 2 ? net->H[l] : nullptr;
        p.ldcb = d[l + 1];
        int rc = l < 2 ? gemm<EPI_BIAS_GELU>(net->stream, p) : gemm<EPI_BIAS>(net->stream, p);
        if (rc) return rc;
        if (l < 2) in = net->H[l];
    }
    return SPDK_OK;
}

// gradients of the MSE loss for B rows (targets T: B x dout, leading dim ldt)
int backward(spdk_mlp* net, int B, const float* T, long ldt) {
    const int* d = net->dims;
    hipStream_t st = net->stream;
    // the gradients of every layer and the loss are one array
    hipLaunchKernelGGL(k_fill, dim3(nb(net->nparam + 1, 256)), dim3(256), 0, st, net->grad, net->nparam + 1, 0.f);
    const float inv = 1.0f / ((float)B * (float)net->dout);
    hipLaunchKernelGGL(k_mse, dim3((d[3] + 255) / 256, (B + kMseRows - 1) / kMseRows), dim3(256), 0, st, net->Z[2],
                       (long)d[3], T, ldt, B, net->dout, d[3], inv, net->dZb[0], net->gb[2], net->loss);
    SPDK_LAUNCH_CHECK("k_mse");
    int cur = 0;
    for (int l = 2; l >= 0; l--) {
        WgradP p{};
        p.dZ = net->dZb[cur];
        p.X = l > 0 ? net->H[l - 1] : net->X;  // layer input (B x d[l])
        p.N = d[l + 1];
        p.K = d[l];
        p.rows = B;
        // rows per workgroup: enough workgroups for the chip, at least 256 rows
        // each (every workgroup adds its 4096 outputs atomically)
        const int tiles = (d[l + 1] / 64) * (d[l] / 64);
        const int split = std::max(1, std::min((B + 255) / 256, (512 + tiles - 1) / tiles));
        p.chunk = ((B + split - 1) / split + TK - 1) / TK * TK;
        p.gW = net->gW[l];
        hipLaunchKernelGGL(k_gemm_wgrad, dim3(d[l] / 64, d[l + 1] / 64, (B + p.chunk - 1) / p.chunk), dim3(256), 0, st, p);
        SPDK_LAUNCH_CHECK("k_gemm_wgrad");
        if (l == 0) break;
        // dH = dZ W (B x d[l]), then dZ_{l-1} = dH * gelu'(Z_{l-1})
        GemmP q{};
        q.A = net->dZb[cur];
        q.lda = d[l + 1];
        q.B = net->WbT[l];  // B(k = out, n = in) = W[out][in] = WbT[in][out]
        q.ldb = d[l + 1];
        q.M = B;
        q.N = d[l];
        q.K = d[l + 1];
        q.Zp = net->Z[l - 1];
        q.ldz = d[l];
        q.Cb = net->dZb[1 - cur];
        q.ldcb = d[l];
        q.colsum = net->gb[l - 1];
        if (int rc = gemm<EPI_GELU_BWD>(st, q)) return rc;
        cur = 1 - cur;
    }
    return SPDK_OK;
}

int check_net(spdk_mlp* net, int B) {
    if (!net) { set_error("mlp: null network"); return SPDK_E_ARG; }
    if (B < 1 || B > net->cap) { set_error("mlp: batch outside 1..capacity"); return SPDK_E_ARG; }
    return SPDK_OK;
}

}  // namespace

extern "C" {

int spdk_mlp_create(const int dims[4], int batch_cap, void* stream, spdk_mlp** out) {
    if (!dims || !out || batch_cap < 1) { set_error("mlp: bad argument"); return SPDK_E_ARG; }
    spdk_mlp* net = new spdk_mlp();
    net->din = dims[0];
    net->dout = dims[3];
    for (int i = 0; i < 4; i++) {
        if (dims[i] < 1 || dims[i] > 65536) { delete net; set_error("mlp: bad dimension"); return SPDK_E_ARG; }
        net->dims[i] = (dims[i] + 63) / 64 * 64;
    }
    net->cap = batch_cap;
    net->stream = (hipStream_t)stream;
    const int* d = net->dims;
    int rc = SPDK_OK;
    auto A = [&](void** p, size_t b) { if (!rc) rc = alloc(net, p, b); };
    int dmax = 0;
    for (int l = 0; l < 3; l++) net->nparam += (long)d[l + 1] * d[l] + d[l + 1];
    A((void**)&net->par, net->nparam * 4);
    A((void**)&net->mom, net->nparam * 4);
    A((void**)&net->var, net->nparam * 4);
    A((void**)&net->grad, (net->nparam + 1) * 4);
    if (!rc) {
        long o = 0;
        for (int l = 0; l < 3; l++) {
            net->W[l] = net->par + o;
            net->gW[l] = net->grad + o;
            o += (long)d[l + 1] * d[l];
            net->b[l] = net->par + o;
            net->gb[l] = net->grad + o;
            o += d[l + 1];
        }
        net->loss = net->grad + net->nparam;
    }
    for (int l = 0; l < 3; l++) {
        size_t nw = (size_t)d[l + 1] * d[l];
        A((void**)&net->Wb[l], nw * 2);
        A((void**)&net->WbT[l], nw * 2);
        A((void**)&net->Z[l], (size_t)batch_cap * d[l + 1] * 4);
        dmax = dmax > d[l + 1] ? dmax : d[l + 1];
    }
    dmax = dmax > d[0] ? dmax : d[0];
    A((void**)&net->X, (size_t)batch_cap * d[0] * 2);
    A((void**)&net->H[0], (size_t)batch_cap * d[1] * 2);
    A((void**)&net->H[1], (size_t)batch_cap * d[2] * 2);
    A((void**)&net->dZb[0], (size_t)batch_cap * dmax * 2);
    A((void**)&net->dZb[1], (size_t)batch_cap * dmax * 2);
    if (rc) { for (void* p : net->owned) (void)hipFree(p); delete net; return rc; }
    *out = net;
    return SPDK_OK;
}

int spdk_mlp_destroy(spdk_mlp* net) {
    if (!net) return SPDK_OK;
    (void)hipStreamSynchronize(net->stream);
    for (void* p : net->owned) (void)hipFree(p);
    delete net;
    return SPDK_OK;
}

int spdk_gather_rows(const float* src, long ld, const int* idx, int n, int cols, float* dst, void* stream) {
    if (!src || !idx || !dst || n < 0 || cols < 0) { set_error("gather: bad argument"); return SPDK_E_ARG; }
    if (n == 0 || cols == 0) return SPDK_OK;
    hipLaunchKernelGGL(k_gather, dim3(nb((long)n * cols, 256)), dim3(256), 0, (hipStream_t)stream, src, ld, idx, n, cols,
                       dst);
    SPDK_LAUNCH_CHECK("k_gather");
    return SPDK_OK;
}

int spdk_rows_finite(const float* Y, long ld, int rows, int cols, float maxabs, unsigned char* flags, void* stream) {
    if (!Y || !flags || rows < 0 || cols < 0) { set_error("rows_finite: bad argument"); return SPDK_E_ARG; }
    if (rows == 0) return SPDK_OK;
    hipLaunchKernelGGL(k_rows_ok, dim3(rows), dim3(256), 0, (hipStream_t)stream, Y, ld, rows, cols, maxabs, flags);
    SPDK_LAUNCH_CHECK("k_rows_ok");
    return SPDK_OK;
}

int spdk_mlp_set_stream(spdk_mlp* net, void* stream) {
    if (!net) return SPDK_E_ARG;
    SPDK_CHECK(hipStreamSynchronize(net->stream));
    net->stream = (hipStream_t)stream;
    return SPDK_OK;
}

int spdk_mlp_dims(spdk_mlp* net, int padded[4]) {
    if (!net || !padded) return SPDK_E_ARG;
    for (int i = 0; i < 4; i++) padded[i] = net->dims[i];
    return SPDK_OK;
}

// Parameters as one FP32 host array, unpadded: W1 (h1 x in), b1, W2, b2, W3, b3.
size_t spdk_mlp_param_count(spdk_mlp* net) {
    if (!net) return 0;
    size_t n = 0;
    const int u[4] = {net->din, net->dims[1], net->dims[2], net->dout};
    for (int l = 0; l < 3; l++) n += (size_t)u[l + 1] * u[l] + u[l + 1];
    return n;
}

static int xfer_params(spdk_mlp* net, float* host, bool to_dev) {
    const int u[4] = {net->din, net->dims[1], net->dims[2], net->dout};
    const int* d = net->dims;
    size_t o = 0;
    for (int l = 0; l < 3; l++) {
        std::vector<float> W((size_t)d[l + 1] * d[l], 0.f), b(d[l + 1], 0.f);
        if (!to_dev) {
            SPDK_CHECK(hipMemcpyAsync(W.data(), net->W[l], W.size() * 4, hipMemcpyDeviceToHost, net->stream));
            SPDK_CHECK(hipMemcpyAsync(b.data(), net->b[l], b.size() * 4, hipMemcpyDeviceToHost, net->stream));
            SPDK_CHECK(hipStreamSynchronize(net->stream));
        }
        for (int r = 0; r < u[l + 1]; r++)
            for (int k = 0; k < u[l]; k++) {
                if (to_dev) W[(size_t)r * d[l] + k] = host[o];
                else host[o] = W[(size_t)r * d[l] + k];
                o++;
            }
        for (int r = 0; r < u[l + 1]; r++) {
            if (to_dev) b[r] = host[o];
            else host[o] = b[r];
            o++;
        }
        if (to_dev) {
            SPDK_CHECK(hipMemcpyAsync(net->W[l], W.data(), W.size() * 4, hipMemcpyHostToDevice, net->stream));
            SPDK_CHECK(hipMemcpyAsync(net->b[l], b.data(), b.size() * 4, hipMemcpyHostToDevice, net->stream));
            const long nw = (long)W.size();
            hipLaunchKernelGGL(k_to_bf16, dim3(nb(nw, 256)), dim3(256), 0, net->stream, (const float*)net->W[l],
                               net->Wb[l], net->WbT[l], nw, d[l], d[l + 1]);
            SPDK_LAUNCH_CHECK("k_to_bf16");
            SPDK_CHECK(hipStreamSynchronize(net->stream));
        }
    }
    return SPDK_OK;
}

int spdk_mlp_set_params(spdk_mlp* net, const float* host) {
    if (!net || !host) return SPDK_E_ARG;
    net->step = 0;
    for (float* p : {net->mom, net->var}) {
        hipLaunchKernelGGL(k_fill, dim3(nb(net->nparam, 256)), dim3(256), 0, net->stream, p, net->nparam, 0.f);
        SPDK_LAUNCH_CHECK("k_fill");
    }
    return xfer_params(net, const_cast<float*>(host), true);
}

int spdk_mlp_get_params(spdk_mlp* net, float* host) {
    if (!net || !host) return SPDK_E_ARG;
    return xfer_params(net, host, false);
}

// Forward pass on B device rows of FP32 features (leading dimension ldx);
// writes the B x dout outputs (leading dimension ldy) to Y (device).
int spdk_mlp_forward(spdk_mlp* net, const float* X, long ldx, int B, float* Y, long ldy) {
    int rc = check_net(net, B);
    if (rc) return rc;
    if (!Y || ldy < net->dout) { set_error("mlp forward: null output or rows shorter than the outputs"); return SPDK_E_ARG; }
    hipLaunchKernelGGL(k_pack_input, dim3(nb((long)B * net->dims[0], 256)), dim3(256), 0, net->stream, X, ldx, B,
                       net->din, net->dims[0], net->X);
    SPDK_LAUNCH_CHECK("k_pack_input");
    return forward(net, B, Y, ldy);
}

// Gradients of the loss mean((f(X) - T)^2) for B device rows, copied to the
// host in the layout of spdk_mlp_set_params; *loss (host) gets the loss.
int spdk_mlp_gradients(spdk_mlp* net, const float* X, long ldx, const float* T, long ldt, int B, float* host_grad,
                       float* loss) {
    int rc = check_net(net, B);
    if (rc) return rc;
    hipLaunchKernelGGL(k_pack_input, dim3(nb((long)B * net->dims[0], 256)), dim3(256), 0, net->stream, X, ldx, B,
                       net->din, net->dims[0], net->X);
    SPDK_LAUNCH_CHECK("k_pack_input");
    if ((rc = forward(net, B))) return rc;
    if ((rc = backward(net, B, T, ldt))) return rc;
    if (loss) {
        SPDK_CHECK(hipMemcpyAsync(loss, net->loss, 4, hipMemcpyDeviceToHost, net->stream));
    }
    SPDK_CHECK(hipStreamSynchronize(net->stream));
    if (host_grad) {
        const int u[4] = {net->din, net->dims[1], net->dims[2], net->dout};
        const int* d = net->dims;
        size_t o = 0;
        for (int l = 0; l < 3; l++) {
            std::vector<float> g((size_t)d[l + 1] * d[l]), gb(d[l + 1]);
            SPDK_CHECK(hipMemcpy(g.data(), net->gW[l], g.size() * 4, hipMemcpyDeviceToHost));
            SPDK_CHECK(hipMemcpy(gb.data(), net->gb[l], gb.size() * 4, hipMemcpyDeviceToHost));
            for (int r = 0; r < u[l + 1]; r++)
                for (int k = 0; k < u[l]; k++) host_grad[o++] = g[(size_t)r * d[l] + k];
            for (int r = 0; r < u[l + 1]; r++) host_grad[o++] = gb[r];
        }
    }
    return SPDK_OK;
}

// One Adam step on B device rows; *loss (host, may be NULL) gets the loss
// before the update (reading it synchronises).
int spdk_mlp_train_step(spdk_mlp* net, const float* X, long ldx, const float* T, long ldt, int B, float lr,
                        float* loss) {
    int rc = check_net(net, B);
    if (rc) return rc;
    hipLaunchKernelGGL(k_pack_input, dim3(nb((long)B * net->dims[0], 256)), dim3(256), 0, net->stream, X, ldx, B,
                       net->din, net->dims[0], net->X);
    SPDK_LAUNCH_CHECK("k_pack_input");
    if ((rc = forward(net, B))) return rc;
    if ((rc = backward(net, B, T, ldt))) return rc;
    net->step++;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float c1 = 1.0f / (1.0f - powf(b1, (float)net->step)), c2 = 1.0f / (1.0f - powf(b2, (float)net->step));
    const int* d = net->dims;
    AdamP p{};
    p.w = net->par;
    p.m = net->mom;
    p.v = net->var;
    p.g = net->grad;
    long o = 0;
    for (int l = 0; l < 3; l++) {
        p.end[2 * l] = o += (long)d[l + 1] * d[l];
        p.end[2 * l + 1] = o += d[l + 1];
        p.rows[l] = d[l + 1];
        p.cols[l] = d[l];
        p.wb[l] = net->Wb[l];
        p.wbT[l] = net->WbT[l];
    }
    p.lr = lr;
    p.b1 = b1;
    p.b2 = b2;
    p.eps = eps;
    p.c1 = c1;
    p.c2 = c2;
    hipLaunchKernelGGL(k_adam, dim3(nb(net->nparam, 256)), dim3(256), 0, net->stream, p);
    SPDK_LAUNCH_CHECK("k_adam");
    if (loss) {
        SPDK_CHECK(hipMemcpyAsync(loss, net->loss, 4, hipMemcpyDeviceToHost, net->stream));
        SPDK_CHECK(hipStreamSynchronize(net->stream));
    }
    return SPDK_OK;
}

}  // extern "C"
