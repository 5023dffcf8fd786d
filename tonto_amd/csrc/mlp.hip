// Training and inference kernels of the learned initial guess's network (FP32).
//
// The products run on the matrix cores (v_mfma_f32_16x16x4f32: FP32 operands, products and
// sums, twice the vector rate without packed FP32), and what bounded the step were its 16
// launches in series, most on 64 work-groups: a 2048-row step of the 273-128-128-225 network
// took 727 us for 0.85 GFLOP.  Now a forward pass is one launch and a backward pass two:
//   forward  16 rows per work-group through all three layers, activations in LDS;
//   chain    16 rows per work-group: dZ2 = (dY W3^T) SiLU'(Z2), dZ1 = (dZ2 W2^T) SiLU'(Z1);
//   weights  32 x 32 tiles of dW1, dW2, dW3 (and the bias sums), eight wavefronts sharing the
//            batch's rows and adding up in LDS: no atomics up to 16384 rows.
// Networks whose 16-row block does not fit the LDS use a general tiled product per layer.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../../include/tonto_mlp.h"

namespace {

struct GemmArgs {
    const float *A;
    long sam, sak;  // A(m, k) = A[m * sam + k * sak]
    const float *B;
    long sbk, sbn;  // B(k, n) = B[k * sbk + n * sbn]
    float *C;
    long scm;       // C(m, n) = C[m * scm + n]
    long M;
    int N, K;
    const float *bias;  // added per column (forward epilogue), or null
    float *Z;           // pre-activation copy (ld scm), or null
    int act;            // 1: SiLU
};

__device__ __forceinline__ float silu(float z) { return z / (1.0f + expf(-z)); }

__device__ __forceinline__ float silu_grad(float z)
{
    const float s = 1.0f / (1.0f + expf(-z));
    return s * (1.0f + z * (1.0f - s));
}

constexpr int TM = 64, TN = 64, TK = 16;

__global__ __launch_bounds__(256) void gemm_kernel(GemmArgs g)
{
    __shared__ float As[TK][TM + 4];
    __shared__ float Bs[TK][TN + 4];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const long m0 = (long)blockIdx.y * TM;
    const int n0 = blockIdx.x * TN;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;
    // lanes walk the unit-stride index of each operand, so tile loads are coalesced
    const bool a_m_fast = g.sam == 1, b_n_fast = g.sbn == 1;
    for (int k0 = 0; k0 < g.K; k0 += TK) {
        for (int t = threadIdx.x; t < TM * TK; t += 256) {
            const int mm = a_m_fast ? t % TM : t / TK, kk = a_m_fast ? t / TM : t % TK;
            const long m = m0 + mm;
            const int k = k0 + kk;
            As[kk][mm] = (m < g.M && k < g.K) ? g.A[m * g.sam + (long)k * g.sak] : 0.0f;
        }
        for (int t = threadIdx.x; t < TN * TK; t += 256) {
            const int nn = b_n_fast ? t % TN : t / TK, kk = b_n_fast ? t / TN : t % TK;
            const int n = n0 + nn, k = k0 + kk;
            Bs[kk][nn] = (n < g.N && k < g.K) ? g.B[(long)k * g.sbk + (long)n * g.sbn] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < TK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const long m = m0 + ty * 4 + i;
        if (m >= g.M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= g.N) continue;
            float v = acc[i][j];
            if (g.bias) v += g.bias[n];
            if (g.Z) g.Z[m * g.scm + n] = v;
            if (g.act) v = silu(v);
            g.C[m * g.scm + n] = v;
        }
    }
}

void gemm(const GemmArgs &g0, hipStream_t s)
{
    const long mt = (g0.M + TM - 1) / TM;
    const int nt = (g0.N + TN - 1) / TN;
    gemm_kernel<<<dim3(nt, (unsigned)mt), 256, 0, s>>>(g0);
}

__global__ void fill_kernel(float *p, long n, float v)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

// d = d * SiLU'(Z)
__global__ void silu_back_kernel(float *d, const float *Z, long n)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        d[i] *= silu_grad(Z[i]);
}

// Work-groups of the loss: each ends in an atomic on the one sum, and those take their turn at
// 14 ns each (1800 work-groups over 4.6e5 outputs: 25 us; 128: 4.5)
constexpr int kLossGroups = 128;

__global__ __launch_bounds__(256) void mse_kernel(const float *Y, const float *T, long n, float scale,
                                                  float *dY, float *loss)
{
    __shared__ float red[256];
    float acc = 0.0f;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const float d = Y[i] - T[i];
        dY[i] = 2.0f * scale * d;
        acc += d * d;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, scale * red[0]);
}

__global__ void adam_kernel(float *p, const float *g, float *m, float *v, long n, float lr, float b1,
                            float b2, float eps, float c1, float c2)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}

// ----------------------------------------------------------------------------------------
// Matrix-core form.  v_mfma_f32_16x16x4f32: lane l gives A(l % 16, l / 16) and B(l / 16, l % 16)
// and holds C(4 (l / 16) + i, l % 16), i = 0 .. 3.
// ----------------------------------------------------------------------------------------
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kRows = 16;    // batch rows of a work-group
constexpr int kWaves = 8;    // wavefronts of a work-group of the gradients
// ... of the forward and chain kernels: the 16 column tiles of 256 hidden units at once (a step
// of 2048 rows, 225 outputs: 81.3 us with 8, 76.9 with 16)
constexpr int kRowWaves = 16;
constexpr int kUnroll = 8;   // k steps (of 4) whose loads are in flight together
constexpr size_t kLdsLimit = 64 * 1024;

// LDS row of K values: zero-padded to whole unrolled steps, odd length (bank spread)
__host__ __device__ constexpr int lds_stride(int K) { return (K + 4 * kUnroll - 1) / (4 * kUnroll) * (4 * kUnroll) + 1; }

// rows m0 .. of the M x K matrix src into LDS (row stride lds_stride(K)), zeros elsewhere
__device__ __forceinline__ void stage_rows(const float *src, long m0, long M, int K, float *dst)
{
    const int s = lds_stride(K);
    for (int t = threadIdx.x; t < kRows * s; t += blockDim.x) {
        const int r = t / s, k = t - r * s;
        dst[t] = k < K && m0 + r < M ? src[(m0 + r) * K + k] : 0.0f;
    }
}

// C = A B for the 16 rows in LDS (As, K columns) and the N columns of B, B(k, n) =
// W[k * sk + n * sn]; done(row, n, value) is called for every element with n < N.
template <typename Done>
__device__ __forceinline__ void rows_product(const float *As, int K, const float *W, long sk, long sn, int N, Done &&done)
{
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const int sa = lds_stride(K);
    for (int t = threadIdx.x >> 6; t * 16 < N; t += kRowWaves) {
        const int n = t * 16 + c;
        const bool in = n < N;
        const float *w = W + (long)(in ? n : 0) * sn;
        f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int k0 = 0; k0 < K; k0 += 4 * kUnroll) {
            float a[kUnroll], b[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const int k = k0 + 4 * u + g;
                a[u] = As[c * sa + k];
                b[u] = in && k < K ? w[(long)k * sk] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b[u], acc, 0, 0, 0);
        }
        if (in) {
#pragma unroll
            for (int i = 0; i < 4; ++i) done(4 * g + i, n, acc[i]);
        }
    }
}

// zero padding of an LDS block whose first N columns rows_product fills
__device__ __forceinline__ void zero_pad(float *dst, int N)
{
    const int s = lds_stride(N), w = s - N;
    for (int t = threadIdx.x; t < kRows * w; t += blockDim.x) dst[t / w * s + N + t % w] = 0.0f;
}

struct NetArgs {
    const float *W1, *b1, *W2, *b2, *W3, *b3;
    int n_in, nh, n_out;
    long M;
};

__host__ __device__ constexpr size_t forward_lds(int n_in, int nh) { return 4u * kRows * ((size_t)lds_stride(n_in) + lds_stride(nh)); }
__host__ __device__ constexpr size_t chain_lds(int nh, int n_out) { return 4u * kRows * ((size_t)lds_stride(n_out) + lds_stride(nh)); }

__global__ __launch_bounds__(64 * kRowWaves) void forward_kernel(NetArgs a, const float *X, float *Z1, float *A1, float *Z2,
                                                             float *A2, float *Y)
{
    extern __shared__ float sm[];
    float *const u = sm, *const v = sm + kRows * (lds_stride(a.n_in) > lds_stride(a.nh) ? lds_stride(a.n_in) : lds_stride(a.nh));
    const long m0 = (long)blockIdx.x * kRows;
    const int sh = lds_stride(a.nh);
    stage_rows(X, m0, a.M, a.n_in, u);
    zero_pad(v, a.nh);
    __syncthreads();
    // one hidden layer: pre-activation and activation out, the activation into LDS too
    auto hidden = [&](const float *b, float *Z, float *A, float *next, int r, int n, float x) {
        const float z = x + b[n], y = silu(z);
        next[r * sh + n] = y;
        if (m0 + r < a.M) {
            Z[(m0 + r) * a.nh + n] = z;
            A[(m0 + r) * a.nh + n] = y;
        }
    };
    rows_product(u, a.n_in, a.W1, a.nh, 1, a.nh, [&](int r, int n, float x) { hidden(a.b1, Z1, A1, v, r, n, x); });
    __syncthreads();
    zero_pad(u, a.nh);  // (u held X)
    rows_product(v, a.nh, a.W2, a.nh, 1, a.nh, [&](int r, int n, float x) { hidden(a.b2, Z2, A2, u, r, n, x); });
    __syncthreads();
    rows_product(u, a.nh, a.W3, a.n_out, 1, a.n_out, [&](int r, int n, float x) {
        if (m0 + r < a.M) Y[(m0 + r) * a.n_out + n] = x + a.b3[n];
    });
}

__global__ __launch_bounds__(64 * kRowWaves) void chain_kernel(NetArgs a, const float *Z1, const float *Z2, const float *dY,
                                                           float *dZ1, float *dZ2)
{
    extern __shared__ float sm[];
    float *const u = sm, *const v = sm + kRows * lds_stride(a.n_out);
    const long m0 = (long)blockIdx.x * kRows;
    const int sh = lds_stride(a.nh);
    stage_rows(dY, m0, a.M, a.n_out, u);
    zero_pad(v, a.nh);
    __syncthreads();
    rows_product(u, a.n_out, a.W3, 1, a.n_out, a.nh, [&](int r, int n, float x) {
        const bool in = m0 + r < a.M;
        const float d = in ? x * silu_grad(Z2[(m0 + r) * a.nh + n]) : 0.0f;
        v[r * sh + n] = d;
        if (in) dZ2[(m0 + r) * a.nh + n] = d;
    });
    __syncthreads();
    rows_product(v, a.nh, a.W2, 1, a.nh, a.nh, [&](int r, int n, float x) {
        if (m0 + r < a.M) dZ1[(m0 + r) * a.nh + n] = x * silu_grad(Z1[(m0 + r) * a.nh + n]);
    });
}

// C(m, n) = sum over the batch of A(r, m) B(r, n), c(n) = sum of B(r, n), three such products;
// a 32 x 32 tile per work-group, the batch's rows shared by its wavefronts (and by gridDim.y
// work-groups, which then add with atomics).
struct GradProduct {
    const float *A, *B;
    float *C, *c;
    int m, n;       // columns of A and of B
    int tn, first;  // tiles along n, first work-group
};
struct GradArgs {
    GradProduct p[3];
    long M;
    long rows;  // batch rows per blockIdx.y, a multiple of 4 kWaves
};

__global__ __launch_bounds__(64 * kWaves) void grad_kernel(GradArgs g)
{
    __shared__ float part[kWaves][32 * 32];
    __shared__ float cpart[kWaves][32];
    const int wg = blockIdx.x;
    const int q = wg >= g.p[2].first ? 2 : wg >= g.p[1].first ? 1 : 0;
    const GradProduct p = g.p[q];
    const int tile = wg - p.first, m0 = tile / p.tn * 32, n0 = tile % p.tn * 32;
    const int lane = threadIdx.x & 63, c = lane & 15, k = lane >> 4, wave = threadIdx.x >> 6;
    const long r_begin = (long)blockIdx.y * g.rows, r_end = min(g.M, r_begin + g.rows);
    const bool ma = m0 + c < p.m, mb = m0 + 16 + c < p.m, na = n0 + c < p.n, nb = n0 + 16 + c < p.n;
    // Sums of kBlock steps (128 rows), added up in `total`.  One FP32 chain over all of a
    // wavefront's rows left a gradient's rms error at 1.9e-7 of its size at 8192 rows, 0.9e-7
    // with blocks (2048 rows: 1.5e-7, 1.3e-7; the step's time is the same).
    constexpr int U = 4, kBlock = 8;
    f4 total[2][2];
    float ctotal[2] = {0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) total[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    f4 acc[2][2];
    float cs[2];
    for (long r0 = r_begin + 4 * U * wave, step = 0; r0 < r_end; r0 += 4 * U * kWaves, ++step) {
        if (step % kBlock == 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (step) total[i][j] += acc[i][j];
                    acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
                }
                if (step) ctotal[i] += cs[i];
                cs[i] = 0.0f;
            }
        }
        float a[U][2], b[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long r = r0 + 4 * u + k;
            const bool in = r < r_end;
            const float *ar = p.A + (in ? r : 0) * p.m + m0 + c, *br = p.B + (in ? r : 0) * p.n + n0 + c;
            a[u][0] = in && ma ? ar[0] : 0.0f;
            a[u][1] = in && mb ? ar[16] : 0.0f;
            b[u][0] = in && na ? br[0] : 0.0f;
            b[u][1] = in && nb ? br[16] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i], b[u][j], acc[i][j], 0, 0, 0);
            cs[0] += b[u][0];
            cs[1] += b[u][1];
        }
    }
    const bool any = r_begin + 4 * U * wave < r_end;  // (else acc and cs are not set)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            if (any) total[i][j] += acc[i][j];
        if (any) ctotal[i] += cs[i];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[wave][(16 * i + 4 * k + e) * 32 + 16 * j + c] = total[i][j][e];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        ctotal[j] += __shfl_xor(ctotal[j], 16, 64);
        ctotal[j] += __shfl_xor(ctotal[j], 32, 64);
        if (k == 0) cpart[wave][16 * j + c] = ctotal[j];
    }
    __syncthreads();
    for (int t = threadIdx.x; t < 32 * 32 + 32; t += 64 * kWaves) {
        const bool bias = t >= 32 * 32;
        const int m = m0 + t / 32, n = n0 + t % 32;
        if (n >= p.n || (bias ? m0 > 0 : m >= p.m)) continue;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) v += bias ? cpart[w][t % 32] : part[w][t];
        float *dst = bias ? p.c + n : p.C + (long)m * p.n + n;
        if (gridDim.y > 1) atomicAdd(dst, v);
        else *dst = v;
    }
}

int grid_1d(long n) { return (int)std::min<long>((n + 255) / 256, 4096); }

struct Layout {
    long W1, b1, W2, b2, W3, b3, n;
};

Layout layout(int n_in, int nh, int n_out)
{
    Layout L;
    L.W1 = 0;
    L.b1 = L.W1 + (long)n_in * nh;
    L.W2 = L.b1 + nh;
    L.b2 = L.W2 + (long)nh * nh;
    L.W3 = L.b2 + nh;
    L.b3 = L.W3 + (long)nh * n_out;
    L.n = L.b3 + n_out;
    return L;
}

// limits: grid.y of the general product holds the row tiles; widths up to 1024
constexpr long kMaxRows = 65535L * TM;

bool bad_dims(int n_in, int nh, int n_out, long M)
{
    return n_in <= 0 || nh <= 0 || n_out <= 0 || M < 0 || M > kMaxRows || nh > 1024 || n_out > 1024 ||
           n_in > (1 << 20);
}

}  // namespace

extern "C" long tmlp_n_params(int n_in, int nh, int n_out) { return layout(n_in, nh, n_out).n; }

extern "C" long tmlp_forward_workspace(long M, int nh) { return 4 * M * (long)nh; }

extern "C" long tmlp_backward_workspace(long M, int nh) { return 2 * M * (long)nh; }

extern "C" int tmlp_forward(const float *params, int n_in, int nh, int n_out, const float *X, long M,
                            float *ws, float *Y, void *stream)
{
    if (!params || !X || !ws || !Y || bad_dims(n_in, nh, n_out, M)) return TMLP_E_ARG;
    if (M == 0) return TMLP_OK;
    hipStream_t s = (hipStream_t)stream;
    const Layout L = layout(n_in, nh, n_out);
    float *Z1 = ws, *A1 = ws + M * nh, *Z2 = ws + 2 * M * nh, *A2 = ws + 3 * M * nh;
    const size_t lds = forward_lds(std::max(n_in, nh), nh);
    if (lds <= kLdsLimit) {
        const NetArgs a{params + L.W1, params + L.b1, params + L.W2, params + L.b2, params + L.W3, params + L.b3, n_in, nh, n_out, M};
        forward_kernel<<<(unsigned)((M + kRows - 1) / kRows), 64 * kRowWaves, lds, s>>>(a, X, Z1, A1, Z2, A2, Y);
        return hipGetLastError() == hipSuccess ? TMLP_OK : TMLP_E_HIP;
    }
    GemmArgs g{};
    g.A = X; g.sam = n_in; g.sak = 1;
    g.B = params + L.W1; g.sbk = nh; g.sbn = 1;
    g.C = A1; g.scm = nh; g.M = M; g.N = nh; g.K = n_in;
    g.bias = params + L.b1; g.Z = Z1; g.act = 1;
    gemm(g, s);
    g.A = A1; g.sam = nh;
    g.B = params + L.W2; g.sbk = nh;
    g.C = A2; g.K = nh; g.bias = params + L.b2; g.Z = Z2;
    gemm(g, s);
    g.A = A2; g.sam = nh;
    g.B = params + L.W3; g.sbk = n_out;
    g.C = Y; g.scm = n_out; g.N = n_out; g.K = nh; g.bias = params + L.b3; g.Z = nullptr; g.act = 0;
    gemm(g, s);
    return hipGetLastError() == hipSuccess ? TMLP_OK : TMLP_E_HIP;
}

extern "C" int tmlp_backward(const float *params, int n_in, int nh, int n_out, const float *X, long M,
                             const float *ws, const float *dY, float *grads, float *ws2, void *stream)
{
    if (!params || !X || !ws || !dY || !grads || !ws2 || bad_dims(n_in, nh, n_out, M)) return TMLP_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    const Layout L = layout(n_in, nh, n_out);
    const long rows_step = 4 * kWaves;
    // one work-group per tile and 16384 rows
    const int kz = (int)std::max(1L, (M + 16383) / 16384);
    if (kz > 1 || M == 0) fill_kernel<<<grid_1d(L.n), 256, 0, s>>>(grads, L.n, 0.0f);
    if (M == 0) return hipGetLastError() == hipSuccess ? TMLP_OK : TMLP_E_HIP;
    const float *Z1 = ws, *A1 = ws + M * nh, *Z2 = ws + 2 * M * nh, *A2 = ws + 3 * M * nh;
    float *dZ1 = ws2, *dZ2 = ws2 + M * nh;
    const size_t lds = chain_lds(nh, n_out);
    if (lds <= kLdsLimit) {
        const NetArgs a{params + L.W1, params + L.b1, params + L.W2, params + L.b2, params + L.W3, params + L.b3, n_in, nh, n_out, M};
        chain_kernel<<<(unsigned)((M + kRows - 1) / kRows), 64 * kRowWaves, lds, s>>>(a, Z1, Z2, dY, dZ1, dZ2);
    } else {
        // dA2 = dY W3^T and dA1 = dZ2 W2^T by the general product, SiLU' in place
        GemmArgs g{};
        g.A = dY; g.sam = n_out; g.sak = 1;
        g.B = params + L.W3; g.sbk = 1; g.sbn = n_out;
        g.C = dZ2; g.scm = nh; g.M = M; g.N = nh; g.K = n_out;
        gemm(g, s);
        silu_back_kernel<<<grid_1d(M * nh), 256, 0, s>>>(dZ2, Z2, M * nh);
        g.A = dZ2; g.sam = nh;
        g.B = params + L.W2; g.sbn = nh;
        g.C = dZ1; g.K = nh;
        gemm(g, s);
        silu_back_kernel<<<grid_1d(M * nh), 256, 0, s>>>(dZ1, Z1, M * nh);
    }
    GradArgs g{};
    g.p[0] = GradProduct{X, dZ1, grads + L.W1, grads + L.b1, n_in, nh, 0, 0};
    g.p[1] = GradProduct{A1, dZ2, grads + L.W2, grads + L.b2, nh, nh, 0, 0};
    g.p[2] = GradProduct{A2, dY, grads + L.W3, grads + L.b3, nh, n_out, 0, 0};
    long tiles = 0;
    for (GradProduct &p : g.p) {
        p.tn = (p.n + 31) / 32;
        p.first = (int)tiles;
        tiles += (long)((p.m + 31) / 32) * p.tn;
    }
    g.M = M;
    g.rows = ((M + kz - 1) / kz + rows_step - 1) / rows_step * rows_step;
    grad_kernel<<<dim3((unsigned)tiles, (unsigned)kz), 64 * kWaves, 0, s>>>(g);
    return hipGetLastError() == hipSuccess ? TMLP_OK : TMLP_E_HIP;
}

extern "C" int tmlp_mse(const float *Y, const float *T, long n, float scale, float *dY, float *loss,
                        void *stream)
{
    if (!Y || !T || !dY || !loss || n < 0) return TMLP_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    fill_kernel<<<1, 64, 0, s>>>(loss, 1, 0.0f);
    if (n) mse_kernel<<<std::min(grid_1d(n), kLossGroups), 256, 0, s>>>(Y, T, n, scale, dY, loss);
    return hipGetLastError() == hipSuccess ? TMLP_OK : TMLP_E_HIP;
}

extern "C" int tmlp_adam(float *params, const float *grads, float *m, float *v, long n, float lr,
                         float beta1, float beta2, float eps, int step, void *stream)
{
    if (!params || !grads || !m || !v || n < 0 || step < 1) return TMLP_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    const float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
    if (n) adam_kernel<<<grid_1d(n), 256, 0, s>>>(params, grads, m, v, n, lr, beta1, beta2, eps, c1, c2);
    return hipGetLastError() == hipSuccess ? TMLP_OK : TMLP_E_HIP;
}
