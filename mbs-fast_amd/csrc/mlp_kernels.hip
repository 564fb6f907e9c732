// mlp_kernels.hip -- the multilayer perceptron of the learned control
// variate: GEMMs on BF16 MFMA with FP32 accumulation (weights and
// activations kept in FP32, rounded to BF16 as they are loaded), exact-erf
// GELU, mean-squared-error gradient, column sums and Adam on FP32 master
// weights.  All kernels are deterministic (no atomics).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mbs {

typedef float mlp_f32x16 __attribute__((ext_vector_type(16)));
typedef short mlp_bf16x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (finite inputs).
__device__ __forceinline__ short to_bf16(float x)
{
    uint32_t u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (short)(u >> 16);
}

// GELU(z) = z Phi(z), Phi the standard normal distribution function.
__device__ __forceinline__ float mlp_gelu(float x)
{
    return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f));
}

// GELU'(z) = Phi(z) + z phi(z).
__device__ __forceinline__ float mlp_gelu_slope(float x)
{
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

// C[M x N] = op(A) op(B), and what follows it: + bias[N]; times GELU'(Z); H =
// GELU(C) beside it.  op(A) is M x K, op(B) K x N.
//   TA = 0: A row-major [M][lda]; TA = 1: A stored [K][lda] (op(A) = A^T)
//   TB = 0: B row-major [K][ldb]; TB = 1: B stored [N][ldb] (op(B) = B^T)
// Products are v_mfma_f32_32x32x8bf16_1k: lane l supplies A[l%32][4(l/32) + q] and
// B[4(l/32) + q][l%32], q = 0..3, for each K step of 8.  K past the end reads as
// zero; rows and columns past the end read the last one, and are not written.
struct MlpGemm {
    int M, N, K;
    const float *A;
    int lda;
    const float *B;
    int ldb;
    float *C;
    int ldc;
    const float *bias;  // [N], or none
    const float *Z;     // [M][ldc], or none
    float *H;           // [M][ldc], or none
};

__device__ __forceinline__ void mlp_store(const MlpGemm &g, int r, int c, float v)
{
    const size_t i = (size_t)r * g.ldc + c;
    v += g.bias ? g.bias[c] : 0.0f;
    if (g.Z)
        v *= mlp_gelu_slope(g.Z[i]);
    g.C[i] = v;
    if (g.H)
        g.H[i] = mlp_gelu(v);
}

// Large products: a workgroup of four waves takes 128 x 128 of C, a wave 64 x 64
// (four accumulators), through LDS tiles of 32 K in BF16; the next tile's loads
// are in flight over this one's products.  The operands pass through L2 once a
// tile, which with C's bytes is the floor (about 25 us of L2 and memory for 4096 x
// 2896 x 256): it takes 54 us there, 80 with the kernel below.
enum { MLP_TILE = 128, MLP_BK = 32, MLP_LD = MLP_BK + 4 };
template <int TA, int TB>
__global__ void __launch_bounds__(256) mlp_tile_kernel(MlpGemm g)
{
    __shared__ __align__(16) short s_a[MLP_TILE][MLP_LD], s_b[MLP_TILE][MLP_LD];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int row0 = blockIdx.y * MLP_TILE, col0 = blockIdx.x * MLP_TILE;
    enum { PER = MLP_TILE * MLP_BK / 256 };  // elements of a tile per thread
    float va[PER], vb[PER];
    // element i of this thread: consecutive threads along the stored rows
    const auto place = [&](int along_k, int i, int &o, int &k) {
        const int e = threadIdx.x + 256 * i;
        o = along_k ? e / MLP_BK : e % MLP_TILE;
        k = along_k ? e % MLP_BK : e / MLP_TILE;
    };
    const auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int o, k;
            place(!TA, i, o, k);
            const int r = min(row0 + o, g.M - 1), ka = min(k0 + k, g.K - 1);
            const float a = TA ? g.A[(size_t)ka * g.lda + r] : g.A[(size_t)r * g.lda + ka];
            va[i] = k0 + k < g.K ? a : 0.0f;
            place(TB, i, o, k);
            const int c = min(col0 + o, g.N - 1), kb = min(k0 + k, g.K - 1);
            const float b = TB ? g.B[(size_t)c * g.ldb + kb] : g.B[(size_t)kb * g.ldb + c];
            vb[i] = k0 + k < g.K ? b : 0.0f;
        }
    };
    mlp_f32x16 acc[2][2] = {};
    const int ar = (w >> 1) * 64 + (lane & 31), bc = (w & 1) * 64 + (lane & 31);
    const int kq = 4 * (lane >> 5);
    load(0);
    for (int k0 = 0; k0 < g.K; k0 += MLP_BK) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            int o, k;
            place(!TA, i, o, k);
            s_a[o][k] = to_bf16(va[i]);
            place(TB, i, o, k);
            s_b[o][k] = to_bf16(vb[i]);
        }
        __syncthreads();
        if (k0 + MLP_BK < g.K)
            load(k0 + MLP_BK);
#pragma unroll
        for (int k = 0; k < MLP_BK; k += 8) {
            mlp_bf16x4 a[2], b[2];
            for (int h = 0; h < 2; ++h) {
                a[h] = *reinterpret_cast<const mlp_bf16x4 *>(&s_a[ar + 32 * h][k + kq]);
                b[h] = *reinterpret_cast<const mlp_bf16x4 *>(&s_b[bc + 32 * h][k + kq]);
            }
            for (int h = 0; h < 2; ++h)
                for (int n = 0; n < 2; ++n)
                    acc[h][n] =
                        __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a[h], b[n], acc[h][n], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
        for (int n = 0; n < 2; ++n)
            for (int v = 0; v < 16; ++v) {
                const int r = row0 + (w >> 1) * 64 + 32 * h + 8 * (v >> 2) + 4 * (lane >> 5) +
                              (v & 3);
                const int c = col0 + bc + 32 * n;
                if (r < g.M && c < g.N)
                    mlp_store(g, r, c, acc[h][n][v]);
            }
}

// The others: a workgroup takes 32 x 32 of C and its waves (SPLIT of them) a share
// of K each, in whole steps; their sums are added in order through LDS.  Operands
// come straight from L2 in groups of 32 K.  SPLIT = 8 keeps a wave from walking a
// long K alone (512 x 256 x 2896: 30 us; 102 in order).  The forward pass takes
// SPLIT = 1: a difference in the last bit of an activation can flip its rounding
// to BF16 in the next layer, so its sums keep the order of K.
template <int TA, int TB, int SPLIT>
__global__ void __launch_bounds__(64 * SPLIT) mlp_split_kernel(MlpGemm g)
{
    __shared__ float s_c[SPLIT > 1 ? SPLIT : 1][16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int row0 = blockIdx.y * 32, col0 = blockIdx.x * 32;
    const int ar = min(row0 + (lane & 31), g.M - 1), bc = min(col0 + (lane & 31), g.N - 1);
    const int kq = 4 * (lane >> 5);
    const int share = ((g.K + SPLIT - 1) / SPLIT + 7) / 8 * 8;
    const int end = min(g.K, share * (w + 1));
    // 16-byte loads along K where rows allow them
    const bool va = !TA && !(g.lda & 3) && !((uintptr_t)g.A & 15);
    const bool vb = TB && !(g.ldb & 3) && !((uintptr_t)g.B & 15);
    // four elements k .. k + 3 of a row of op(A) or column of op(B)
    const auto quad = [&](const float *p, int ld, int o, bool along, bool wide, int k) {
        float4 f;
        if (wide) {
            f = *reinterpret_cast<const float4 *>(p + (size_t)o * ld + k);
        } else {
            f.x = along ? p[(size_t)o * ld + k] : p[(size_t)k * ld + o];
            f.y = along ? p[(size_t)o * ld + k + 1] : p[(size_t)(k + 1) * ld + o];
            f.z = along ? p[(size_t)o * ld + k + 2] : p[(size_t)(k + 2) * ld + o];
            f.w = along ? p[(size_t)o * ld + k + 3] : p[(size_t)(k + 3) * ld + o];
        }
        return f;
    };
    const auto round4 = [](float4 f) {
        return mlp_bf16x4{to_bf16(f.x), to_bf16(f.y), to_bf16(f.z), to_bf16(f.w)};
    };
    mlp_f32x16 acc = {};
    int k0 = share * w;
    for (; k0 + 32 <= end; k0 += 32) {
        float4 a[4], b[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            a[u] = quad(g.A, g.lda, ar, !TA, va, k0 + 8 * u + kq);
            b[u] = quad(g.B, g.ldb, bc, TB, vb, k0 + 8 * u + kq);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(round4(a[u]), round4(b[u]), acc, 0, 0, 0);
    }
    for (; k0 < end; k0 += 8) {
        mlp_bf16x4 a, b;
        for (int q = 0; q < 4; ++q) {
            const int k = min(k0 + kq + q, g.K - 1);
            const float x = TA ? g.A[(size_t)k * g.lda + ar] : g.A[(size_t)ar * g.lda + k];
            const float y = TB ? g.B[(size_t)bc * g.ldb + k] : g.B[(size_t)k * g.ldb + bc];
            a[q] = k0 + kq + q < end ? to_bf16(x) : (short)0;
            b[q] = k0 + kq + q < end ? to_bf16(y) : (short)0;
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, acc, 0, 0, 0);
    }
    if constexpr (SPLIT == 1) {
        for (int v = 0; v < 16; ++v) {
            const int r = row0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
            if (r < g.M && col0 + (lane & 31) < g.N)
                mlp_store(g, r, col0 + (lane & 31), acc[v]);
        }
        return;
    }
    for (int v = 0; v < 16; ++v)
        s_c[w][v][lane] = acc[v];
    __syncthreads();
    for (int i = threadIdx.x; i < 1024; i += 64 * SPLIT) {
        const int v = i >> 6, l = i & 63;
        const int r = row0 + 8 * (v >> 2) + 4 * (l >> 5) + (v & 3), c = col0 + (l & 31);
        float sum = s_c[0][v][l];
        for (int e = 1; e < SPLIT; ++e)
            sum += s_c[e][v][l];
        if (r < g.M && c < g.N)
            mlp_store(g, r, c, sum);
    }
}

// dY = 2 (Y - T) / (rows * cols); per-row partial sums of (Y - T)^2.
__global__ void mlp_mse_grad_kernel(int rows, int cols, const float *__restrict__ y,
                                    const float *__restrict__ t, float *__restrict__ dy,
                                    float *__restrict__ row_sq)
{
    const int r = blockIdx.x;
    const float scale = 2.0f / ((float)rows * (float)cols);
    float s = 0.0f;
    for (int c = threadIdx.x; c < cols; c += blockDim.x) {
        const size_t i = (size_t)r * cols + c;
        const float d = y[i] - t[i];
        dy[i] = scale * d;
        s += d * d;
    }
    __shared__ float red[256];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = blockDim.x / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o)
            red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        row_sq[r] = red[0];
}

// out[c] = sum over rows of m[r][c]: 32 columns and 16 slices of the rows a
// workgroup, the slices' sums added in order.  One thread a column waited for
// 512 rows one after the other: 109 us, now 3 to 4.
enum { COLSUM_SLICES = 16 };
__global__ void __launch_bounds__(32 * COLSUM_SLICES)
    mlp_colsum_kernel(int rows, int cols, const float *__restrict__ m, float *__restrict__ out)
{
    __shared__ float s_sum[COLSUM_SLICES][32];
    const int l = threadIdx.x & 31, slice = threadIdx.x >> 5;
    const int c = min((int)blockIdx.x * 32 + l, cols - 1);
    const int end = (int)((int64_t)rows * (slice + 1) / COLSUM_SLICES);
    float s = 0.0f;
    int r = (int)((int64_t)rows * slice / COLSUM_SLICES);
    for (; r + 8 <= end; r += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            v[u] = m[(size_t)(r + u) * cols + c];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            s += v[u];
    }
    for (; r < end; ++r)
        s += m[(size_t)r * cols + c];
    s_sum[slice][l] = s;
    __syncthreads();
    if (slice == 0 && (int)blockIdx.x * 32 + l < cols) {
        for (int e = 1; e < COLSUM_SLICES; ++e)
            s += s_sum[e][l];
        out[c] = s;
    }
}

// Adam (bias-corrected), FP32 master weights.
__global__ void mlp_adam_kernel(size_t n, float *__restrict__ w, const float *__restrict__ g,
                                float *__restrict__ m, float *__restrict__ v, float lr,
                                float b1, float b2, float eps, float c1, float c2)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// Gathers rows idx[0..rows) of src [*, cols] into dst [rows, cols].
__global__ void mlp_gather_kernel(int rows, int cols, const int32_t *__restrict__ idx,
                                  const float *__restrict__ src, float *__restrict__ dst)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)rows * cols)
        return;
    const int r = (int)(i / cols), c = (int)(i - (size_t)r * cols);
    dst[i] = src[(size_t)idx[r] * cols + c];
}

}  // namespace mbs
