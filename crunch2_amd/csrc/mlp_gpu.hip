// mlp_gpu.hip -- learned DXT1 endpoint proposal: features, training kernels,
// BF16 matrix-core inference and the integer refinement that judges it.
//
// No reference counterpart: the learned proposal sits beside crnlib's
// dxt1_endpoint_optimizer (crnlib/crn_dxt1.cpp:2234).  The features restate the
// block statistics of compute_vectors / compute_pca (crn_dxt1.cpp:155-256); the
// refinement is the +-1 endpoint lattice of refine_solution / the 26-neighbour
// probe (crn_dxt1.cpp:601-643, 905-1016) judged by the exact DXT1 block error
// (crn_dxt1.cpp:1370-1592, weights 8/25/1 from crn_color.h:724-726).
//
// Model: 57 -> 128 -> 128 -> 7, tanh-form GELU, weights and layer inputs in
// bfloat16, sums in float32.  Training is one fused kernel for the batch's loss
// and gradient and Adam; the layer-by-layer pieces (a strided FP32 GEMM with
// bf16 rounding of the operands on load, bias/GELU and loss kernels) stand as
// entry points of their own; inference is one fused kernel on
// v_mfma_f32_32x32x16_bf16 (a wave owns 32 blocks, weights staged in LDS).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>

#include "crn2_internal.h"

namespace {

constexpr uint32_t kIn = 57, kHid = 128, kOut = 7;
constexpr float kGeluC = 0.7978845608028654f;
constexpr float kGeluA = 0.044715f;
constexpr float kConfWeight = 0.05f;

__device__ inline float bf16_round(float x)
{
    uint32_t u = __float_as_uint(x);
    u = (u + 0x7FFFu + ((u >> 16) & 1u)) & 0xFFFF0000u;
    return __uint_as_float(u);
}

__device__ inline float gelu(float z)
{
    const float t = tanhf(kGeluC * (z + kGeluA * z * z * z));
    return 0.5f * z * (1.0f + t);
}

__device__ inline float gelu_grad(float z)
{
    const float t = tanhf(kGeluC * (z + kGeluA * z * z * z));
    const float du = kGeluC * (1.0f + 3.0f * kGeluA * z * z);
    return 0.5f * (1.0f + t) + 0.5f * z * (1.0f - t * t) * du;
}

// ------------------------------------------------------------- features
__device__ inline void block_features(const uint8_t* px, float* f)
{
    float c[16][3];
    float mean[3] = {0, 0, 0};
    for (int p = 0; p < 16; p++)
        for (int k = 0; k < 3; k++) {
            c[p][k] = (float)px[4 * p + k] / 255.0f;
            mean[k] += c[p][k];
        }
    for (int k = 0; k < 3; k++) mean[k] /= 16.0f;
    for (int p = 0; p < 16; p++)
        for (int k = 0; k < 3; k++) f[3 * p + k] = c[p][k] - 0.5f;
    for (int i = 0; i < 3; i++)
        for (int jj = 0; jj < 3; jj++) {
            float s = 0;
            for (int p = 0; p < 16; p++) s += (c[p][i] - mean[i]) * (c[p][jj] - mean[jj]);
            f[48 + 3 * i + jj] = s / 16.0f * 4.0f;
        }
}

__global__ void __launch_bounds__(256) mlp_features_kernel(const uint8_t* __restrict__ rgba, uint32_t n,
                                                           float* __restrict__ feat)
{
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= n) return;
    block_features(rgba + (size_t)b * 64, feat + (size_t)b * kIn);
}

// ---------------------------------------------------------------- GEMM
// C(m, n) [+]= sum_k A(m, k) B(k, n), A(m, k) = A[m sam + k sak],
// B(k, n) = B[k sbk + n sbn], C row-major with leading dimension ldc.  64 x 64
// tiles, 16-deep K slices in LDS, 4 x 4 outputs per thread; grid.z splits K
// and adds its partial sums atomically (C must then start cleared).
struct GemmArgs {
    const float* A;
    const float* B;
    float* C;
    uint32_t M, N, K;
    int64_t sam, sak, sbk, sbn, ldc;
    int accumulate;      // add into C instead of overwriting it
    int round_a, round_b;
};

__global__ void __launch_bounds__(256) gemm_f32_kernel(GemmArgs g)
{
    __shared__ float As[16][64 + 1];
    __shared__ float Bs[16][64 + 1];
    const uint32_t tid = threadIdx.x;
    const uint32_t tx = tid & 15u, ty = tid >> 4;
    const uint32_t m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    const uint32_t ksplit = (g.K + gridDim.z - 1) / gridDim.z;
    const uint32_t kb = blockIdx.z * ksplit, ke = min(g.K, kb + ksplit);
    float acc[4][4] = {};
    for (uint32_t k0 = kb; k0 < ke; k0 += 16) {
        for (uint32_t e = tid; e < 1024; e += 256) {
            const uint32_t kk = e >> 6, mm = e & 63u;
            const uint32_t m = m0 + mm, k = k0 + kk;
            float a = 0, b = 0;
            if (m < g.M && k < ke) {
                a = g.A[(int64_t)m * g.sam + (int64_t)k * g.sak];
                if (g.round_a) a = bf16_round(a);
            }
            const uint32_t nn = n0 + mm;
            if (nn < g.N && k < ke) {
                b = g.B[(int64_t)k * g.sbk + (int64_t)nn * g.sbn];
                if (g.round_b) b = bf16_round(b);
            }
            As[kk][mm] = a;
            Bs[kk][mm] = b;
        }
        __syncthreads();
#pragma unroll
        for (uint32_t kk = 0; kk < 16; kk++) {
            float a[4], b[4];
            for (int i = 0; i < 4; i++) a[i] = As[kk][ty * 4 + i];
            for (int i = 0; i < 4; i++) b[i] = Bs[kk][tx * 4 + i];
            for (int i = 0; i < 4; i++)
                for (int jj = 0; jj < 4; jj++) acc[i][jj] = fmaf(a[i], b[jj], acc[i][jj]);
        }
        __syncthreads();
    }
    for (int i = 0; i < 4; i++) {
        const uint32_t m = m0 + ty * 4 + i;
        if (m >= g.M) continue;
        for (int jj = 0; jj < 4; jj++) {
            const uint32_t nn = n0 + tx * 4 + jj;
            if (nn >= g.N) continue;
            float* c = g.C + (int64_t)m * g.ldc + nn;
            if (gridDim.z > 1) atomicAdd(c, acc[i][jj]);
            else *c = g.accumulate ? *c + acc[i][jj] : acc[i][jj];
        }
    }
}

// ------------------------------------------------- bias, activation, loss
// Z = C + bias (row broadcast); with gelu, A = bf16(gelu(Z)), else A = Z.
__global__ void __launch_bounds__(256) bias_act_kernel(float* __restrict__ Z, float* __restrict__ A,
                                                       const float* __restrict__ bias, uint32_t rows, uint32_t cols,
                                                       int use_gelu)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (uint64_t)rows * cols) return;
    const float z = Z[i] + bias[i % cols];
    Z[i] = z;
    A[i] = use_gelu ? bf16_round(gelu(z)) : z;
}

__global__ void __launch_bounds__(256) gelu_back_kernel(const float* __restrict__ dA, const float* __restrict__ Z,
                                                        float* __restrict__ dZ, uint64_t n)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dZ[i] = dA[i] * gelu_grad(Z[i]);
}

// Y: rows x 7 outputs, T: rows x 6 targets.  dY = d loss / dY for the batch
// mean of squared error (outputs 0-5) + kConfWeight * logistic loss of
// output 6 against "all six rounded components within one step".
__global__ void __launch_bounds__(256) mlp_loss_kernel(const float* __restrict__ Y, const float* __restrict__ T,
                                                       const float* __restrict__ labels, uint32_t rows,
                                                       float* __restrict__ dY, float* __restrict__ loss)
{
    __shared__ float red[256];
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0;
    if (r < rows) {
        const float* y = Y + (size_t)r * kOut;
        const float* t = T + (size_t)r * 6;
        const float scale[6] = {31, 63, 31, 31, 63, 31};
        bool ok = true;
        const float inv = 1.0f / (float)rows;
        for (int k = 0; k < 6; k++) {
            const float d = y[k] - t[k];
            l += d * d;
            dY[(size_t)r * kOut + k] = 2.0f * inv * d;
            const float q = fminf(fmaxf(rintf(y[k] * scale[k]), 0.0f), scale[k]);
            ok &= fabsf(q - rintf(t[k] * scale[k])) <= 1.0f;
        }
        const float lab = labels ? labels[r] : (ok ? 1.0f : 0.0f);
        const float z = y[6];
        const float s = 1.0f / (1.0f + expf(-z));
        l += kConfWeight * (fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z))) - lab * z);
        dY[(size_t)r * kOut + 6] = kConfWeight * inv * (s - lab);
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (uint32_t s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, red[0] / (float)rows);
}

// ------------------------------------------------- fused training gradient
// Loss and gradient of a batch in one pass over its rows: a workgroup of four
// waves takes R rows at a time through forward, loss and backward with every
// layer in LDS or registers, keeps its part of the gradient in registers over
// all its rows, and writes it once; mlp_grad_reduce_kernel adds the
// workgroups' parts in a fixed order.
//   forward: bfloat16 operands on v_mfma_f32_32x32x16_bf16; wave w computes
//     columns 32 w .. of a layer and keeps gelu'(z) of its outputs;
//   backward: float32 operands on v_mfma_f32_32x32x2_f32 (the gradients stay
//     in float32, the bfloat16-rounded weights and activations are exact in
//     it); the product's layout is that of the kept gelu'(z).
// X carries a column of ones behind its 57 features (its weights are zero), so
// that layer 1's bias gradient is a row of its weight gradient.
// What bounds it: the float32 matrix products (64 cycles each) of the four
// waves of each CU.  As 15 launches of a strided vector GEMM and elementwise
// kernels 32,768 rows took 1,290 us, now 80 us (262,144 rows: 6,194, now 523).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr uint32_t kInPad = 64;               // K of layer 1 (57 features + zeros)
constexpr uint32_t kOutPad = 32;              // N of layer 3 (7 outputs + zeros)
constexpr uint32_t kXs = kInPad + 8;          // LDS row strides (bf16 elements), padded against bank conflicts
constexpr uint32_t kHs = kHid + 8;
constexpr uint32_t kParams = kIn * kHid + kHid + kHid * kHid + kHid + kHid * kOut + kOut;
constexpr uint32_t kPartial = kParams + 1;    // a workgroup's part: the gradient, then the loss
constexpr uint32_t kDzs = kHid + 5;           // float row stride: an odd step between rows and columns alike
constexpr uint32_t kMaxGradWgs = 256;

__device__ inline bf16x8 lds_bf16x8(const uint8_t* lds, uint32_t byte_ofs)
{
    return *reinterpret_cast<const bf16x8*>(lds + byte_ofs);
}

__device__ inline __bf16 to_bf16(float x)
{
    const uint32_t u = __float_as_uint(bf16_round(x)) >> 16;
    return __builtin_bit_cast(__bf16, (uint16_t)u);
}

__device__ inline float from_bf16(__bf16 x)
{
    return __uint_as_float((uint32_t)__builtin_bit_cast(uint16_t, x) << 16);
}

template <uint32_t R>
struct GradLds {
    __bf16 w1[kHid][kXs];       // W1 transposed: [n][k]
    __bf16 w2[kHid][kHs];
    __bf16 w3[kOutPad][kHs];
    float bias[2 * kHid + 8];
    __bf16 x[R][kXs];
    __bf16 a1[R][kHs];
    __bf16 a2[R][kHs];
    float y[R][8];              // outputs, then their gradient
    float dz[R][kDzs];
};

// gelu and its derivative from one tanh
__device__ inline void gelu_both(float z, float& a, float& g)
{
    const float t = tanhf(kGeluC * (z + kGeluA * z * z * z));
    const float du = kGeluC * (1.0f + 3.0f * kGeluA * z * z);
    a = 0.5f * z * (1.0f + t);
    g = 0.5f * (1.0f + t) + 0.5f * z * (1.0f - t * t) * du;
}

// One layer's columns c0 .. c0 + 31 of R rows: z = in W + b, its activation
// into `out` and gelu'(z) into g (row 32 m + 8 (i / 4) + 4 half + i % 4 of
// register i).
template <uint32_t R, uint32_t KS>
__device__ inline void grad_layer(const __bf16* in, uint32_t is, const __bf16* w, uint32_t ws, const float* bias,
                                  uint32_t c0, __bf16 (*out)[kHs], float (*g)[16])
{
    const uint32_t lane = threadIdx.x & 63u, half = lane >> 5, col = lane & 31u;
    f32x16 acc[R / 32];
#pragma unroll
    for (uint32_t m = 0; m < R / 32; m++) acc[m] = f32x16{0};
#pragma unroll
    for (uint32_t ks = 0; ks < KS; ks++) {
        const uint32_t k = 16 * ks + 8 * half;
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(w + (c0 + col) * ws + k);
#pragma unroll
        for (uint32_t m = 0; m < R / 32; m++) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(in + (32 * m + col) * is + k);
            acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[m], 0, 0, 0);
        }
    }
    const float bc = bias[c0 + col];
#pragma unroll
    for (uint32_t m = 0; m < R / 32; m++)
#pragma unroll
        for (uint32_t i = 0; i < 16; i++) {
            float act;
            gelu_both(acc[m][i] + bc, act, g[m][i]);
            out[32 * m + 8 * (i >> 2) + 4 * half + (i & 3)][c0 + col] = to_bf16(act);
        }
}

template <uint32_t R>
__global__ void __launch_bounds__(256) mlp_grad_kernel(const float* __restrict__ X, const float* __restrict__ T,
                                                       const float* __restrict__ labels, uint32_t rows,
                                                       const float* __restrict__ theta, float* __restrict__ part)
{
    extern __shared__ __align__(16) uint8_t lds[];
    GradLds<R>& L = *reinterpret_cast<GradLds<R>*>(lds);
    constexpr uint32_t M = R / 32;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, half = lane >> 5, col = lane & 31u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), c0 = 32 * wave;
    const float* W1 = theta;
    const float* b1 = W1 + kIn * kHid;
    const float* W2 = b1 + kHid;
    const float* b2 = W2 + kHid * kHid;
    const float* W3 = b2 + kHid;
    const float* b3 = W3 + kHid * kOut;
    // weights (bf16, transposed so that a column is contiguous in K)
#pragma unroll 8
    for (uint32_t e = tid; e < kIn * kHid; e += 256) L.w1[e & 127u][e >> 7] = to_bf16(W1[e]);
    for (uint32_t e = tid; e < (kXs - kIn) * kHid; e += 256) L.w1[e & 127u][kIn + (e >> 7)] = to_bf16(0.0f);
#pragma unroll 8
    for (uint32_t e = tid; e < kHid * kHid; e += 256) L.w2[e & 127u][e >> 7] = to_bf16(W2[e]);
    for (uint32_t e = tid; e < kOutPad * kHs; e += 256) {
        const uint32_t o = e / kHs, k = e % kHs;
        L.w3[o][k] = to_bf16(k < kHid && o < kOut ? W3[k * kOut + o] : 0.0f);
    }
    for (uint32_t e = tid; e < 2 * kHid + 8; e += 256)
        L.bias[e] = e < kHid ? b1[e] : e < 2 * kHid ? b2[e - kHid] : (e - 2 * kHid < kOut ? b3[e - 2 * kHid] : 0.0f);

    f32x16 g1[2], g2[4], g3;     // gradient tiles: W1 (both k tiles) x columns c0, W2 k tile c0 x all, W3 k tile c0
#pragma unroll
    for (uint32_t t = 0; t < 2; t++) g1[t] = f32x16{0};
#pragma unroll
    for (uint32_t t = 0; t < 4; t++) g2[t] = f32x16{0};
    g3 = f32x16{0};
    float db2 = 0.0f, db3 = 0.0f, loss = 0.0f;
    const float inv = 1.0f / (float)rows;
    const uint32_t tiles = (rows + R - 1) / R;
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint32_t r0 = tile * R;
        __syncthreads();   // the previous tile's last reads (and the weights)
#pragma unroll 4
        for (uint32_t e = tid; e < R * kInPad; e += 256) {
            const uint32_t r = e >> 6, k = e & 63u;
            const float v = k < kIn && r0 + r < rows ? X[(size_t)(r0 + r) * kIn + k] : (k == kIn ? 1.0f : 0.0f);
            L.x[r][k] = to_bf16(v);
        }
        __syncthreads();
        float p1[M][16], p2[M][16];
        grad_layer<R, kInPad / 16>(&L.x[0][0], kXs, &L.w1[0][0], kXs, L.bias, c0, L.a1, p1);
        __syncthreads();
        grad_layer<R, kHid / 16>(&L.a1[0][0], kHs, &L.w2[0][0], kHs, L.bias + kHid, c0, L.a2, p2);
        __syncthreads();
        if (wave < M) {
            f32x16 acc = {0};
#pragma unroll
            for (uint32_t ks = 0; ks < kHid / 16; ks++) {
                const uint32_t k = 16 * ks + 8 * half;
                const bf16x8 a = *reinterpret_cast<const bf16x8*>(&L.a2[32 * wave + col][k]);
                const bf16x8 b = *reinterpret_cast<const bf16x8*>(&L.w3[col][k]);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
            }
            if (col < 8) {
                const float bc = L.bias[2 * kHid + col];
#pragma unroll
                for (uint32_t i = 0; i < 16; i++) L.y[32 * wave + 8 * (i >> 2) + 4 * half + (i & 3)][col] = acc[i] + bc;
            }
        }
        __syncthreads();
        // the loss and its gradient, one row per lane (mlp_loss_kernel's formulas)
        if (tid < R) {
            const uint32_t r = r0 + tid;
            float dy[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            if (r < rows) {
                const float scale[6] = {31, 63, 31, 31, 63, 31};
                bool ok = true;
                for (int k = 0; k < 6; k++) {
                    const float y = L.y[tid][k], t = T[(size_t)r * 6 + k];
                    const float d = y - t;
                    loss += d * d;
                    dy[k] = 2.0f * inv * d;
                    const float q = fminf(fmaxf(rintf(y * scale[k]), 0.0f), scale[k]);
                    ok &= fabsf(q - rintf(t * scale[k])) <= 1.0f;
                }
                const float lab = labels ? labels[r] : (ok ? 1.0f : 0.0f);
                const float z = L.y[tid][6];
                const float sg = 1.0f / (1.0f + expf(-z));
                loss += kConfWeight * (fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z))) - lab * z);
                dy[6] = kConfWeight * inv * (sg - lab);
            }
            for (int k = 0; k < 8; k++) L.y[tid][k] = dy[k];
        }
        __syncthreads();
        // dA2 = dY W3^T, dZ2 = dA2 gelu'(Z2)
#pragma unroll
        for (uint32_t m = 0; m < M; m++) {
            f32x16 acc = {0};
#pragma unroll
            for (uint32_t o = 0; o < 8; o += 2)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(L.y[32 * m + col][o + half],
                                                           from_bf16(L.w3[o + half][c0 + col]), acc, 0, 0, 0);
#pragma unroll
            for (uint32_t i = 0; i < 16; i++)
                L.dz[32 * m + 8 * (i >> 2) + 4 * half + (i & 3)][c0 + col] = acc[i] * p2[m][i];
        }
        // dW3 and db3
#pragma unroll 8
        for (uint32_t r = 0; r < R; r += 2)
            g3 = __builtin_amdgcn_mfma_f32_32x32x2f32(from_bf16(L.a2[r + half][c0 + col]),
                                                      col < 8 ? L.y[r + half][col & 7u] : 0.0f, g3, 0, 0, 0);
        if (tid >= 128 && tid < 128 + kOut)
            for (uint32_t r = 0; r < R; r++) db3 += L.y[r][tid - 128];
        __syncthreads();
        // dW2 and db2
#pragma unroll 4
        for (uint32_t r = 0; r < R; r += 2) {
            const float a = from_bf16(L.a1[r + half][c0 + col]);
#pragma unroll
            for (uint32_t t = 0; t < 4; t++)
                g2[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, L.dz[r + half][32 * t + col], g2[t], 0, 0, 0);
        }
        if (tid < kHid)
            for (uint32_t r = 0; r < R; r++) db2 += L.dz[r][tid];
        // dA1 = dZ2 W2^T, dZ1 = dA1 gelu'(Z1)
        {
            f32x16 acc[M];
#pragma unroll
            for (uint32_t m = 0; m < M; m++) acc[m] = f32x16{0};
#pragma unroll 8
            for (uint32_t n = 0; n < kHid; n += 2) {
                const float b = from_bf16(L.w2[n + half][c0 + col]);
#pragma unroll
                for (uint32_t m = 0; m < M; m++)
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(L.dz[32 * m + col][n + half], b, acc[m], 0, 0, 0);
            }
            __syncthreads();   // dZ2 has been read
#pragma unroll
            for (uint32_t m = 0; m < M; m++)
#pragma unroll
                for (uint32_t i = 0; i < 16; i++)
                    L.dz[32 * m + 8 * (i >> 2) + 4 * half + (i & 3)][c0 + col] = acc[m][i] * p1[m][i];
        }
        __syncthreads();
        // dW1, and db1 in row 57
#pragma unroll 4
        for (uint32_t r = 0; r < R; r += 2) {
            const float b = L.dz[r + half][c0 + col];
#pragma unroll
            for (uint32_t t = 0; t < 2; t++)
                g1[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(from_bf16(L.x[r + half][32 * t + col]), b, g1[t], 0, 0, 0);
        }
    }
    // this workgroup's part, laid out as the parameters
    float* P = part + (size_t)blockIdx.x * kPartial;
#pragma unroll
    for (uint32_t i = 0; i < 16; i++) {
        const uint32_t row = 8 * (i >> 2) + 4 * half + (i & 3);
#pragma unroll
        for (uint32_t t = 0; t < 2; t++) {
            const uint32_t k = 32 * t + row;
            if (k <= kIn) P[k * kHid + c0 + col] = g1[t][i];   // row 57: b1 follows W1
        }
#pragma unroll
        for (uint32_t t = 0; t < 4; t++) P[(kIn + 1) * kHid + (c0 + row) * kHid + 32 * t + col] = g2[t][i];
        if (col < kOut) P[(kIn + 2 + kHid) * kHid + (c0 + row) * kOut + col] = g3[i];
    }
    if (tid < kHid) P[(kIn + 1 + kHid) * kHid + tid] = db2;
    if (tid >= 128 && tid < 128 + kOut) P[kParams - kOut + tid - 128] = db3;
    if (tid < 64) {
        for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off);
        if (tid == 0) P[kParams] = loss;
    }
}

// Sums of the workgroups' parts, in order within each of four quarters; the
// last sum is the loss over the batch.
__global__ void __launch_bounds__(256) mlp_grad_reduce_kernel(const float* __restrict__ part, uint32_t n,
                                                              float* __restrict__ g, float* __restrict__ loss,
                                                              uint32_t rows)
{
    __shared__ float s[4][64];
    const uint32_t q = threadIdx.x >> 6, lane = threadIdx.x & 63u, e = blockIdx.x * 64 + lane;
    const uint32_t per = (n + 3) / 4, k0 = min(q * per, n), k1 = min(k0 + per, n);
    float v = 0.0f;
    if (e < kPartial) {
#pragma unroll 8
        for (uint32_t k = k0; k < k1; k++) v += part[(size_t)k * kPartial + e];
    }
    s[q][lane] = v;
    __syncthreads();
    if (q == 0 && e < kPartial) {
        const float t = (s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]);
        if (e < kParams) g[e] = t;
        else *loss = t / (float)rows;
    }
}

// Rows per workgroup step: 32 while that still leaves CUs without work at 64.
inline uint32_t grad_rows(uint32_t n) { return n <= 32 * kMaxGradWgs ? 32u : 64u; }
inline uint32_t grad_wgs(uint32_t n)
{
    return std::min<uint32_t>(kMaxGradWgs, (uint32_t)(((uint64_t)n + grad_rows(n) - 1) / grad_rows(n)));
}

__global__ void __launch_bounds__(256) adam_kernel(float* __restrict__ w, const float* __restrict__ g,
                                                   float* __restrict__ m, float* __restrict__ v, uint32_t n, float lr,
                                                   float b1, float b2, float eps, float c1, float c2)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ------------------------------------------------- matrix-core inference
constexpr uint32_t kInferWaves = 4;
// LDS layout (bytes)
constexpr uint32_t kW1Ofs = 0;                                    // [128][kXs]  W1 transposed (n-major, k contiguous)
constexpr uint32_t kW2Ofs = kW1Ofs + kHid * kXs * 2;              // [128][kHs]
constexpr uint32_t kW3Ofs = kW2Ofs + kHid * kHs * 2;              // [32][kHs]
constexpr uint32_t kBOfs = kW3Ofs + kOutPad * kHs * 2;            // biases: 128 + 128 + 32 floats
constexpr uint32_t kWaveOfs = kBOfs + (2 * kHid + kOutPad) * 4;   // per wave: two [32][kHs] buffers
constexpr uint32_t kWaveBytes = 2 * 32 * kHs * 2;
constexpr uint32_t kInferLds = kWaveOfs + kInferWaves * kWaveBytes;

// One layer for the wave's 32 rows: in [32][ks] bf16 (row stride `is`), out
// written as bf16(gelu(z)) into [32][os] or, for the last layer, z to `y`.
template <uint32_t KSTEPS, uint32_t NTILES, bool LAST>
__device__ inline void mfma_layer(const uint8_t* lds, uint32_t in_ofs, uint32_t is, uint32_t w_ofs, uint32_t ws,
                                  const float* bias, uint8_t* out_lds, uint32_t out_ofs, uint32_t os, float* y,
                                  uint32_t row0, uint32_t n)
{
    const uint32_t lane = threadIdx.x & 63u, g = lane >> 5, col = lane & 31u;
    for (uint32_t nt = 0; nt < NTILES; nt++) {
        f32x16 acc = {0};
#pragma unroll
        for (uint32_t ks = 0; ks < KSTEPS; ks++) {
            const uint32_t k = 16 * ks + 8 * g;
            const bf16x8 a = lds_bf16x8(lds, in_ofs + (col * is + k) * 2);
            const bf16x8 b = lds_bf16x8(lds, w_ofs + ((32 * nt + col) * ws + k) * 2);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
        }
        const uint32_t c = 32 * nt + col;
        const float bc = bias[c];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t r = 8 * (i >> 2) + 4 * g + (i & 3);
            const float z = acc[i] + bc;
            if (LAST) {
                if (c < kOut && row0 + r < n) y[(size_t)(row0 + r) * 8 + c] = z;
            } else {
                *reinterpret_cast<__bf16*>(out_lds + out_ofs + (r * os + c) * 2) = to_bf16(gelu(z));
            }
        }
    }
}

__global__ void __launch_bounds__(256) mlp_infer_kernel(const uint8_t* __restrict__ rgba, uint32_t n,
                                                        const float* __restrict__ theta, float* __restrict__ y)
{
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t tid = threadIdx.x;
    // stage weights (bf16, transposed so a column of W is contiguous in K)
    const float* W1 = theta;
    const float* b1 = W1 + kIn * kHid;
    const float* W2 = b1 + kHid;
    const float* b2 = W2 + kHid * kHid;
    const float* W3 = b2 + kHid;
    const float* b3 = W3 + kHid * kOut;
    for (uint32_t e = tid; e < kHid * kXs; e += 256) {
        const uint32_t nn = e / kXs, k = e % kXs;
        reinterpret_cast<__bf16*>(lds + kW1Ofs)[e] = to_bf16(k < kIn ? W1[k * kHid + nn] : 0.0f);
    }
    for (uint32_t e = tid; e < kHid * kHs; e += 256) {
        const uint32_t nn = e / kHs, k = e % kHs;
        reinterpret_cast<__bf16*>(lds + kW2Ofs)[e] = to_bf16(k < kHid ? W2[k * kHid + nn] : 0.0f);
    }
    for (uint32_t e = tid; e < kOutPad * kHs; e += 256) {
        const uint32_t nn = e / kHs, k = e % kHs;
        reinterpret_cast<__bf16*>(lds + kW3Ofs)[e] = to_bf16(k < kHid && nn < kOut ? W3[k * kOut + nn] : 0.0f);
    }
    float* bl = reinterpret_cast<float*>(lds + kBOfs);
    for (uint32_t e = tid; e < 2 * kHid + kOutPad; e += 256)
        bl[e] = e < kHid ? b1[e] : e < 2 * kHid ? b2[e - kHid] : (e - 2 * kHid < kOut ? b3[e - 2 * kHid] : 0.0f);
    __syncthreads();

    const uint32_t wave = tid >> 6, lane = tid & 63u;
    const uint32_t bufA = kWaveOfs + wave * kWaveBytes, bufB = bufA + 32 * kHs * 2;
    const uint32_t tiles = (n + 31) / 32;
    for (uint32_t t = blockIdx.x * kInferWaves + wave; t < tiles; t += gridDim.x * kInferWaves) {
        const uint32_t row0 = t * 32;
        // features of the wave's 32 blocks into bufA as [32][kXs] bf16 (lanes 0-31, one block each)
        if (lane < 32) {
            float f[kIn];
            const uint32_t b = row0 + lane;
            if (b < n) block_features(rgba + (size_t)b * 64, f);
            else
                for (uint32_t k = 0; k < kIn; k++) f[k] = 0;
            __bf16* xr = reinterpret_cast<__bf16*>(lds + bufA) + lane * kXs;
            for (uint32_t k = 0; k < kInPad; k++) xr[k] = to_bf16(k < kIn ? f[k] : 0.0f);
        }
        __builtin_amdgcn_wave_barrier();
        mfma_layer<kInPad / 16, kHid / 32, false>(lds, bufA, kXs, kW1Ofs, kXs, bl, lds, bufB, kHs, nullptr, row0, n);
        __builtin_amdgcn_wave_barrier();
        mfma_layer<kHid / 16, kHid / 32, false>(lds, bufB, kHs, kW2Ofs, kHs, bl + kHid, lds, bufA, kHs, nullptr, row0,
                                                n);
        __builtin_amdgcn_wave_barrier();
        mfma_layer<kHid / 16, 1, true>(lds, bufA, kHs, kW3Ofs, kHs, bl + 2 * kHid, nullptr, 0, 0, y, row0, n);
        __builtin_amdgcn_wave_barrier();
    }
}

// --------------------------------------------------------- refinement
__device__ inline void expand565(uint32_t c, int* o)
{
    const int r = (c >> 11) & 31, g = (c >> 5) & 63, b = c & 31;
    o[0] = (r << 3) | (r >> 2);
    o[1] = (g << 2) | (g >> 4);
    o[2] = (b << 3) | (b >> 2);
}

// Exact perceptual error of the DXT1 block (c0, c1) with best selectors under
// the standard DXT1 decode: c0 > c1 four colours, c0 <= c1 three + black.
__device__ inline uint32_t dxt1_error(const int (*px)[3], uint32_t c0, uint32_t c1, uint32_t* sel_out)
{
    int p[4][3];
    expand565(c0, p[0]);
    expand565(c1, p[1]);
    const bool four = c0 > c1;
    for (int k = 0; k < 3; k++) {
        if (four) {
            p[2][k] = (2 * p[0][k] + p[1][k]) / 3;
            p[3][k] = (p[0][k] + 2 * p[1][k]) / 3;
        } else {
            p[2][k] = (p[0][k] + p[1][k]) / 2;
            p[3][k] = 0;
        }
    }
    uint32_t err = 0, sel = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        uint32_t best = 0xFFFFFFFFu, bs = 0;
        for (int s = 0; s < 4; s++) {
            const int dr = px[i][0] - p[s][0], dg = px[i][1] - p[s][1], db = px[i][2] - p[s][2];
            const uint32_t e = (uint32_t)(8 * dr * dr + 25 * dg * dg + db * db);
            if (e < best) {
                best = e;
                bs = (uint32_t)s;
            }
        }
        err += best;
        sel |= bs << (2 * i);
    }
    if (sel_out) *sel_out = sel;
    return err;
}

__device__ inline uint32_t pack565(const int* c) { return ((uint32_t)c[0] << 11) | ((uint32_t)c[1] << 5) | (uint32_t)c[2]; }

// The same error, but stops summing once it reaches `bound` (returns a value
// >= bound then): a candidate that cannot win costs only a few texels.
__device__ inline uint32_t dxt1_error_below(const int (*px)[3], uint32_t c0, uint32_t c1, uint32_t bound)
{
    int p[4][3];
    expand565(c0, p[0]);
    expand565(c1, p[1]);
    const bool four = c0 > c1;
    for (int k = 0; k < 3; k++) {
        if (four) {
            p[2][k] = (2 * p[0][k] + p[1][k]) / 3;
            p[3][k] = (p[0][k] + 2 * p[1][k]) / 3;
        } else {
            p[2][k] = (p[0][k] + p[1][k]) / 2;
            p[3][k] = 0;
        }
    }
    uint32_t err = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        uint32_t best = 0xFFFFFFFFu;
        for (int s = 0; s < 4; s++) {
            const int dr = px[i][0] - p[s][0], dg = px[i][1] - p[s][1], db = px[i][2] - p[s][2];
            best = min(best, (uint32_t)(8 * dr * dr + 25 * dg * dg + db * db));
        }
        err += best;
        if (err >= bound) break;
    }
    return err;
}

// Ordered-pair error of (a, b) as pair_error, bounded as dxt1_error_below.
__device__ inline uint32_t pair_error_below(const int (*px)[3], const int* a, const int* b, uint32_t bound)
{
    const uint32_t ca = pack565(a), cb = pack565(b);
    return dxt1_error_below(px, ca > cb ? ca : cb, ca > cb ? cb : ca, bound);
}

// Four-colour error of the unordered endpoint pair (a, b) (equal pairs use the
// three-colour decode); returns the ordered pair in (lo, hi).
__device__ inline uint32_t pair_error(const int (*px)[3], const int* a, const int* b, uint32_t& lo, uint32_t& hi)
{
    const uint32_t ca = pack565(a), cb = pack565(b);
    lo = ca > cb ? ca : cb;
    hi = ca > cb ? cb : ca;
    return dxt1_error(px, lo, hi, nullptr);
}

// +-1 single-channel steps from endpoints e while the exact error drops.
// Returns true if it stopped at a point no single step improves.
__device__ inline bool descend(const int (*px)[3], int (*e)[3], uint32_t& best, uint32_t max_iters, uint32_t& steps)
{
    const int lim[3] = {31, 63, 31};
    for (;;) {
        if (steps >= max_iters) return false;
        uint32_t cand = best;
        int bs = -1, bk = 0, bd = 0;
        for (int s = 0; s < 2; s++)
            for (int k = 0; k < 3; k++)
                for (int d = -1; d <= 1; d += 2) {
                    const int v = e[s][k] + d;
                    if (v < 0 || v > lim[k]) continue;
                    e[s][k] = v;
                    const uint32_t er = pair_error_below(px, e[0], e[1], cand);
                    e[s][k] = v - d;
                    if (er < cand) {
                        cand = er;
                        bs = s;
                        bk = k;
                        bd = d;
                    }
                }
        if (bs < 0) return true;
        for (int s = 0; s < 2; s++)      // static indices: e stays in registers
            for (int k = 0; k < 3; k++)
                if (s == bs && k == bk) e[s][k] += bd;
        best = cand;
        steps++;
    }
}

// Least-squares endpoints for the selectors of the four-colour block (lo, hi)
// (colour i = lo + w_i (hi - lo), w in {0, 1/3, 2/3, 1}), per channel in
// 8-bit space, rounded to 5:6:5.  False if the selectors use one weight only.
__device__ inline bool lsq_endpoints(const int (*px)[3], uint32_t lo, uint32_t hi, int (*e)[3])
{
    uint32_t sel;
    dxt1_error(px, lo, hi, &sel);
    const int u_of[4] = {0, 3, 1, 2};   // 3 w by selector
    int a11 = 0, a12 = 0, a22 = 0, b1[3] = {0, 0, 0}, b2[3] = {0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int u = u_of[(sel >> (2 * i)) & 3u], v = 3 - u;
        a11 += v * v;
        a12 += u * v;
        a22 += u * u;
        for (int k = 0; k < 3; k++) {
            b1[k] += v * px[i][k];
            b2[k] += u * px[i][k];
        }
    }
    const float det = (float)a11 * (float)a22 - (float)a12 * (float)a12;
    if (det <= 0.0f) return false;
    const float lim[3] = {31.0f, 63.0f, 31.0f};
    for (int k = 0; k < 3; k++) {
        const float A = 3.0f * ((float)a22 * (float)b1[k] - (float)a12 * (float)b2[k]) / det;
        const float B = 3.0f * ((float)a11 * (float)b2[k] - (float)a12 * (float)b1[k]) / det;
        e[0][k] = (int)fminf(fmaxf(rintf(A * lim[k] / 255.0f), 0.0f), lim[k]);
        e[1][k] = (int)fminf(fmaxf(rintf(B * lim[k] / 255.0f), 0.0f), lim[k]);
    }
    return true;
}

// Descent, then while the least-squares refit of the result's selectors
// lowers the error, descent again from the refit.
__device__ inline uint32_t refine_from(const int (*px)[3], int (*e)[3], uint32_t max_iters, bool refit,
                                       uint32_t& steps)
{
    uint32_t lo, hi;
    uint32_t best = pair_error(px, e[0], e[1], lo, hi);
    uint32_t used = 0;
    for (int round = 0;; round++) {
        if (!descend(px, e, best, max_iters, used) || !refit || round == 3) break;
        pair_error(px, e[0], e[1], lo, hi);
        if (lo == hi) break;
        int f[2][3];
        if (!lsq_endpoints(px, lo, hi, f)) break;
        const uint32_t ef = pair_error(px, f[0], f[1], lo, hi);
        if (ef >= best) break;
        best = ef;
        for (int s = 0; s < 2; s++)
            for (int k = 0; k < 3; k++) e[s][k] = f[s][k];
    }
    steps += used;
    return best;
}

// Principal-axis start: the extreme projections of the texels on the
// dominant eigenvector of their covariance (power iteration).
__device__ inline void pca_start(const int (*px)[3], int (*e)[3])
{
    float m[3] = {0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; i++)
        for (int k = 0; k < 3; k++) m[k] += (float)px[i][k];
    for (int k = 0; k < 3; k++) m[k] *= 1.0f / 16.0f;
    float c[6] = {0, 0, 0, 0, 0, 0};   // xx xy xz yy yz zz
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float x = px[i][0] - m[0], y = px[i][1] - m[1], z = px[i][2] - m[2];
        c[0] += x * x;
        c[1] += x * y;
        c[2] += x * z;
        c[3] += y * y;
        c[4] += y * z;
        c[5] += z * z;
    }
    float v[3] = {1.0f, 1.0f, 1.0f};
    for (int it = 0; it < 8; it++) {
        const float a = c[0] * v[0] + c[1] * v[1] + c[2] * v[2];
        const float b = c[1] * v[0] + c[3] * v[1] + c[4] * v[2];
        const float d = c[2] * v[0] + c[4] * v[1] + c[5] * v[2];
        const float mx = fmaxf(fabsf(a), fmaxf(fabsf(b), fabsf(d)));
        if (mx <= 0.0f) break;
        v[0] = a / mx;
        v[1] = b / mx;
        v[2] = d / mx;
    }
    const float n2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
    float tmin = 0.0f, tmax = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float t = ((px[i][0] - m[0]) * v[0] + (px[i][1] - m[1]) * v[1] + (px[i][2] - m[2]) * v[2]) / n2;
        tmin = fminf(tmin, t);
        tmax = fmaxf(tmax, t);
    }
    const float lim[3] = {31.0f, 63.0f, 31.0f};
    for (int k = 0; k < 3; k++) {
        e[0][k] = (int)fminf(fmaxf(rintf((m[k] + tmax * v[k]) * lim[k] / 255.0f), 0.0f), lim[k]);
        e[1][k] = (int)fminf(fmaxf(rintf((m[k] + tmin * v[k]) * lim[k] / 255.0f), 0.0f), lim[k]);
    }
}

__device__ inline void net_start(const float* y, int (*e)[3])
{
    const float lim[3] = {31.0f, 63.0f, 31.0f};
    for (int s = 0; s < 2; s++)
        for (int k = 0; k < 3; k++) e[s][k] = (int)fminf(fmaxf(rintf(y[3 * s + k] * lim[k]), 0.0f), lim[k]);
}

// Brightest and darkest texels (first extreme), kept by value so that the
// texels are only ever indexed statically.
__device__ inline void box_start(const int (*px)[3], int (*e)[3])
{
    int bl = -1, dl = 1 << 30, bc[3] = {0, 0, 0}, dc[3] = {0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int l = 2 * px[i][0] + 4 * px[i][1] + px[i][2];
        if (l > bl) {
            bl = l;
            for (int k = 0; k < 3; k++) bc[k] = px[i][k];
        }
        if (l < dl) {
            dl = l;
            for (int k = 0; k < 3; k++) dc[k] = px[i][k];
        }
    }
    const float lim[3] = {31.0f, 63.0f, 31.0f};
    for (int k = 0; k < 3; k++) {
        e[0][k] = (int)rintf((float)bc[k] * lim[k] / 255.0f);
        e[1][k] = (int)rintf((float)dc[k] * lim[k] / 255.0f);
    }
}

// Start points, each refined, the lowest final error kept (earlier start on
// ties): bit 0 of `starts` = the network's proposal y (8 floats per block,
// components scaled to [0, 1]); bit 1 = the block's brightest and darkest
// texels (luma 2r + 4g + b, first extreme); bit 2 = the principal axis.
// Bit 3 adds the least-squares refit after each descent; with bit 4 (the
// both-ends lattice, polish_kernel) the steps carry kSwapped when the second
// endpoint packs higher.
// out per block (16 bytes): u32 c0 | c1 << 16, u32 selectors, u32 error,
// u32 single steps taken (max_iters per start = stopped early)
constexpr uint32_t kSwapped = 1u << 31;

__global__ void __launch_bounds__(256) refine_kernel(const uint8_t* __restrict__ rgba, uint32_t n,
                                                     const float* __restrict__ y, uint32_t max_iters, uint32_t starts,
                                                     uint32_t* __restrict__ out)
{
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= n) return;
    int px[16][3];
#pragma unroll
    for (int i = 0; i < 16; i++)
        for (int k = 0; k < 3; k++) px[i][k] = rgba[(size_t)b * 64 + 4 * i + k];
    const bool refit = (starts & 8u) != 0;
    uint32_t best = 0xFFFFFFFFu, steps = 0;
    int keep[2][3] = {{0, 0, 0}, {0, 0, 0}};
    auto consider = [&](int (*e)[3]) {
        uint32_t st = 0;
        const uint32_t eb = refine_from(px, e, max_iters, refit, st);
        steps = max(steps, st);
        if (eb < best) {
            best = eb;
            for (int s = 0; s < 2; s++)
                for (int k = 0; k < 3; k++) keep[s][k] = e[s][k];
        }
    };
    int e[2][3];
    if (starts & 1u) {
        net_start(y + (size_t)b * 8, e);
        consider(e);
    }
    if (starts & 2u) {
        box_start(px, e);
        consider(e);
    }
    if (starts & 4u) {
        pca_start(px, e);
        consider(e);
    }
    uint32_t lo, hi, sel;
    pair_error(px, keep[0], keep[1], lo, hi);
    best = dxt1_error(px, lo, hi, &sel);
    // the polish goes on from the endpoints in their own order
    if ((starts & 16u) && pack565(keep[0]) < pack565(keep[1])) steps |= kSwapped;
    out[(size_t)b * 4 + 0] = lo | (hi << 16);
    out[(size_t)b * 4 + 1] = sel;
    out[(size_t)b * 4 + 2] = best;
    out[(size_t)b * 4 + 3] = steps;
}

// ------------------------------------------------------------------ polish
// Best improving move among all 728 combinations of -1 / 0 / +1 on the six
// endpoint components (refine_solution's both-ends lattice,
// crnlib/crn_dxt1.cpp:601-643), up to four times, each followed by the
// single-step descent (and refit); one wavefront per block.
//
// A candidate's palette is separable: every channel has nine (low, high)
// moves, and a texel's distance to entry s is the sum of three per-channel
// terms w (p^2 - 2 p c) (the texel's own w c^2 is the same for all).  The terms
// are a product on the matrix cores, exact as in the cluster search: integers
// of at most 8 significant bits times powers of two in bfloat16, sums below
// 2^24 in float32.  K slots 0-7 hold red, 8-15 green, 16-23 blue, so that a
// lane loads its 16 bytes of a candidate's row from a table of 3 x 9 moves, and
// one v_mfma_f32_16x16x32_bf16 gives 4 candidates x 4 entries x 16 texels.
// Red and green alone (81 moves) bound the whole error from below, with the
// smallest blue error added; only moves whose bound is below the best are
// scored in full.  Ties go to the lowest move number, the order of the
// reference's loops.  Candidates with equal endpoints decode as three colours
// and black and are scored on the side.
// What bounds it: the vector operations around each product (minimum, sum over
// 16 lanes).  One lane per block scanning 728 candidates took most of the
// refinement's 7.04 ms for 262,144 blocks; both kernels together now 2.01 ms.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct PolishLds {
    u32x4 row[3][9][4];      // channel, move, entry: 8 bfloat16
    u32x4 zero;
    uint32_t rg[84];         // error of red and green
    uint32_t blue[12];       // error of blue
    uint32_t list[732];      // candidates: moves of the channels (4 bits each) | number << 16
};

__device__ inline uint32_t bf2(float a, float b)
{
    return (__float_as_uint(a) >> 16) | (__float_as_uint(b) & 0xFFFF0000u);
}

__device__ inline uint32_t lane_value(uint32_t v, uint32_t l) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l); }

template <int Ctrl>
__device__ inline uint32_t dpp_of(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, Ctrl, 0xF, 0xF, false);
}

// Sum over the 16 lanes of a row, on each of them.
__device__ inline uint32_t row_sum(uint32_t v)
{
    v += dpp_of<0x128>(v);   // row_ror 8, 4, 2, 1
    v += dpp_of<0x124>(v);
    v += dpp_of<0x122>(v);
    return v + dpp_of<0x121>(v);
}

__device__ inline uint32_t wave_min(uint32_t v)
{
    v = min(v, dpp_of<0x128>(v));
    v = min(v, dpp_of<0x124>(v));
    v = min(v, dpp_of<0x122>(v));
    v = min(v, dpp_of<0x121>(v));
    return min(min(lane_value(v, 0), lane_value(v, 16)), min(lane_value(v, 32), lane_value(v, 48)));
}

// The block on a wave: lane l holds texel l & 15 in `own` and texels
// 4 (l & 3) .. + 3 in `quad` (r | g << 8 | b << 16).
struct WaveBlock {
    uint32_t own, quad[4];
};

struct Ends {
    int e[2][3];
};

__device__ inline uint32_t colour_distance(uint32_t px, const int* p)
{
    const int dr = (int)(px & 255u) - p[0], dg = (int)((px >> 8) & 255u) - p[1], db = (int)((px >> 16) & 255u) - p[2];
    return (uint32_t)(8 * dr * dr + 25 * dg * dg + db * db);
}

// dxt1_error's palette of the unordered pair (a, b).
__device__ inline void pair_palette(const int* a, const int* b, int (*p)[3])
{
    const uint32_t ca = pack565(a), cb = pack565(b);
    const bool four = ca != cb;
    expand565(max(ca, cb), p[0]);
    expand565(min(ca, cb), p[1]);
    for (int k = 0; k < 3; k++) {
        p[2][k] = four ? (2 * p[0][k] + p[1][k]) / 3 : (p[0][k] + p[1][k]) / 2;
        p[3][k] = four ? (p[0][k] + 2 * p[1][k]) / 3 : 0;
    }
}

// Error of each quad's pair (the same on its four lanes).
__device__ inline uint32_t quad_error(const WaveBlock& B, const int* a, const int* b)
{
    int p[4][3];
    pair_palette(a, b, p);
    uint32_t err = 0;
#pragma unroll
    for (int j = 0; j < 4; j++)
        err += min(min(colour_distance(B.quad[j], p[0]), colour_distance(B.quad[j], p[1])),
                   min(colour_distance(B.quad[j], p[2]), colour_distance(B.quad[j], p[3])));
    err += dpp_of<0xB1>(err);   // quad_perm 1 0 3 2
    return err + dpp_of<0x4E>(err);   // quad_perm 2 3 0 1
}

// Selector of the lane's own texel under pair (a, b).
__device__ inline uint32_t own_selector(const WaveBlock& B, const int* a, const int* b)
{
    int p[4][3];
    pair_palette(a, b, p);
    uint32_t best = 0xFFFFFFFFu, s = 0;
    for (uint32_t t = 0; t < 4; t++) {
        const uint32_t e = colour_distance(B.own, p[t]);
        if (e < best) {
            best = e;
            s = t;
        }
    }
    return s;
}

// descend() on a wave: the twelve steps of an iteration on a quad each.
__device__ inline bool wave_descend(const WaveBlock& B, Ends& E, uint32_t& best, uint32_t max_iters, uint32_t& steps)
{
    const uint32_t c = (threadIdx.x & 63u) >> 2;
    for (;;) {
        if (steps >= max_iters) return false;
        int f[2][3];
        bool ok = c < 12;
        for (uint32_t s = 0; s < 2; s++)
            for (uint32_t k = 0; k < 3; k++) {
                f[s][k] = E.e[s][k] + (c >> 1 == 3 * s + k ? ((c & 1u) ? 1 : -1) : 0);
                ok &= f[s][k] >= 0 && f[s][k] <= (k == 1 ? 63 : 31);
            }
        const uint32_t er = quad_error(B, f[0], f[1]);   // out of range: not taken
        const uint32_t m = wave_min(ok && er < best ? er << 4 | c : 0xFFFFFFFFu);
        if (m == 0xFFFFFFFFu) return true;
        const uint32_t t = m & 15u;
        for (uint32_t s = 0; s < 2; s++)
            for (uint32_t k = 0; k < 3; k++) E.e[s][k] += t >> 1 == 3 * s + k ? ((t & 1u) ? 1 : -1) : 0;
        best = m >> 4;
        steps++;
    }
}

// lsq_endpoints() on a wave (four-colour pairs: a != b).
__device__ inline bool wave_lsq(const WaveBlock& B, const Ends& E, Ends& F)
{
    const uint32_t sel = own_selector(B, E.e[0], E.e[1]);
    const uint32_t u = sel == 0 ? 0u : sel == 1 ? 3u : sel == 2 ? 1u : 2u, v = 3u - u;
    const float a11 = (float)(int)lane_value(row_sum(v * v), 0), a12 = (float)(int)lane_value(row_sum(u * v), 0),
                a22 = (float)(int)lane_value(row_sum(u * u), 0);
    const float det = a11 * a22 - a12 * a12;
    if (!(det > 0.0f)) return false;
    const float lim[3] = {31.0f, 63.0f, 31.0f};
    for (int k = 0; k < 3; k++) {
        const uint32_t x = (B.own >> (8 * k)) & 255u;
        const float b1 = (float)(int)lane_value(row_sum(v * x), 0), b2 = (float)(int)lane_value(row_sum(u * x), 0);
        const float A = 3.0f * (a22 * b1 - a12 * b2) / det;
        const float C = 3.0f * (a11 * b2 - a12 * b1) / det;
        F.e[0][k] = (int)fminf(fmaxf(rintf(A * lim[k] / 255.0f), 0.0f), lim[k]);
        F.e[1][k] = (int)fminf(fmaxf(rintf(C * lim[k] / 255.0f), 0.0f), lim[k]);
    }
    return true;
}

// refine_from() on a wave.
__device__ inline uint32_t wave_refine(const WaveBlock& B, Ends& E, uint32_t max_iters, bool refit, uint32_t& steps)
{
    uint32_t best = lane_value(quad_error(B, E.e[0], E.e[1]), 0), used = 0;
    for (int round = 0;; round++) {
        if (!wave_descend(B, E, best, max_iters, used) || !refit || round == 3) break;
        if (pack565(E.e[0]) == pack565(E.e[1])) break;
        Ends F;
        if (!wave_lsq(B, E, F)) break;
        const uint32_t ef = lane_value(quad_error(B, F.e[0], F.e[1]), 0);
        if (ef >= best) break;
        best = ef;
        E = F;
    }
    steps = max(steps, used);
    return best;
}

// Sums over the texels of the smallest entry distances (without the texels'
// own w c^2) of the product of a row operand with the texels: lane group g's
// candidate on its 16 lanes.
__device__ inline int product_error(const u32x4& a, const u32x4& texels)
{
    typedef __bf16 b8 __attribute__((ext_vector_type(8)));
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, texels),
                                                            zero, 0, 0, 0);
    return (int)row_sum((uint32_t)(int)fminf(fminf(d[0], d[1]), fminf(d[2], d[3])));
}

// One lattice step from E: true (E and best updated) if some move improves.
__device__ inline bool wave_box_step(PolishLds& L, const WaveBlock& B, const u32x4& texels, int own_rg, int own_b,
                                     Ends& E, uint32_t& best)
{
    const uint32_t lane = threadIdx.x & 63u, group = lane >> 4;
    // the table: one move and entry of a channel per lane and turn
    __builtin_amdgcn_wave_barrier();   // the last step's has been read
    for (uint32_t i = lane; i < 3 * 9 * 4; i += 64) {
        const uint32_t ch = i / 36, mv = i / 4 % 9, entry = i & 3u;
        const int e0 = (ch == 0 ? E.e[0][0] : ch == 1 ? E.e[0][1] : E.e[0][2]) + (int)(mv % 3) - 1;
        const int e1 = (ch == 0 ? E.e[1][0] : ch == 1 ? E.e[1][1] : E.e[1][2]) + (int)(mv / 3) - 1;
        const int c0 = min(max(e0, 0), ch == 1 ? 63 : 31), c1 = min(max(e1, 0), ch == 1 ? 63 : 31);
        const int p0 = ch == 1 ? (c0 << 2) | (c0 >> 4) : (c0 << 3) | (c0 >> 2);
        const int p1 = ch == 1 ? (c1 << 2) | (c1 >> 4) : (c1 << 3) | (c1 >> 2);
        const int p = entry == 0 ? p0 : entry == 1 ? p1 : entry == 2 ? (2 * p0 + p1) / 3 : (p0 + 2 * p1) / 3;
        const uint32_t K = (ch == 0 ? 8u : ch == 1 ? 25u : 1u) * (uint32_t)(p * p);
        const float f = (float)p, k2 = (float)(K & 0xFF0000u), k1 = (float)(K & 0xFF00u), k0 = (float)(K & 0xFFu);
        u32x4 v;
        if (ch == 1) v = u32x4{bf2(-32.0f * f, -16.0f * f), bf2(-2.0f * f, k2), bf2(k1, k0), 0u};
        else v = u32x4{bf2(ch == 0 ? -16.0f * f : -2.0f * f, k2), bf2(k1, k0), 0u, 0u};
        L.row[ch][mv][entry] = v;
    }
    __builtin_amdgcn_wave_barrier();
    const uint32_t cand = (lane & 15u) >> 2, entry = lane & 3u;   // of the lane's operand row
    // blue alone, then red and green
    for (uint32_t i = 0; i < 12; i += 4) {
        const int e = product_error(group == 2 ? L.row[2][min(i + cand, 8u)][entry] : L.zero, texels) + own_b;
        if ((lane & 15u) == 0) L.blue[i + group] = (uint32_t)e;
    }
    for (uint32_t i = 0; i < 84; i += 4) {
        const uint32_t c = min(i + cand, 80u);
        const int e = product_error(group == 0 ? L.row[0][c % 9][entry] : group == 1 ? L.row[1][c / 9][entry] : L.zero,
                                    texels) + own_rg;
        if ((lane & 15u) == 0) L.rg[i + group] = (uint32_t)e;
    }
    __builtin_amdgcn_wave_barrier();
    // which moves keep a channel in range: bits 0-8 per channel
    uint32_t in[3];
    for (uint32_t k = 0; k < 3; k++) {
        const int lim = k == 1 ? 63 : 31;
        const uint32_t a = (E.e[0][k] > 0 ? 1u : 0u) | 2u | (E.e[0][k] < lim ? 4u : 0u);
        in[k] = (E.e[1][k] > 0 ? a : 0u) | (a << 3) | (E.e[1][k] < lim ? a << 6 : 0u);
    }
    const uint32_t blue = lane < 9 && (in[2] >> lane & 1u) ? L.blue[min(lane, 8u)] : 0xFFFFFFFFu;
    const uint32_t least_blue = wave_min(blue);
    // moves that make a channel's two values equal
    uint32_t eq[3];
    for (uint32_t k = 0; k < 3; k++) {
        eq[k] = 0;
        for (uint32_t mv = 0; mv < 9; mv++)
            eq[k] |= E.e[0][k] + (int)(mv % 3) == E.e[1][k] + (int)(mv / 3) ? 1u << mv : 0u;
    }
    // candidates: the red and green moves below the best, each with the nine blue ones
    uint32_t count = 0;
    for (uint32_t i0 = 0; i0 < 81; i0 += 64) {
        const uint32_t i = min(i0 + lane, 80u), r = i % 9, g = i / 9;
        uint64_t keep = __ballot(i0 + lane < 81 && (in[0] >> r & 1u) && (in[1] >> g & 1u) && L.rg[i] + least_blue < best);
        while (keep) {
            const uint32_t c = i0 + (uint32_t)__builtin_ctzll(keep);
            keep &= keep - 1;
            const uint32_t r9 = c % 9, g9 = c / 9, b9 = min(lane, 8u);
            const uint32_t number = r9 % 3 + 3 * (g9 % 3) + 9 * (b9 % 3) + 27 * (r9 / 3) + 81 * (g9 / 3) + 243 * (b9 / 3);
            const bool same = (eq[0] >> r9 & 1u) && (eq[1] >> g9 & 1u) && (eq[2] >> b9 & 1u);
            const bool ok = lane < 9 && (in[2] >> b9 & 1u) && !same && number != 364 && L.rg[c] + blue < best;
            const uint64_t mask = __ballot(ok);
            if (ok) L.list[count + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = r9 | g9 << 4 | b9 << 8 | number << 16;
            count += (uint32_t)__popcll(mask);
        }
    }
    __builtin_amdgcn_wave_barrier();
    uint32_t least = best, which = 0xFFFFFFFFu;
    for (uint32_t i = 0; i < count; i += 4) {
        const uint32_t c = L.list[min(i + cand, count - 1)], mine = L.list[min(i + group, count - 1)];
        const u32x4 a = group < 3 ? L.row[group][(c >> (4 * group)) & 15u][entry] : L.zero;
        const uint32_t e = (uint32_t)(product_error(a, texels) + own_rg + own_b), number = mine >> 16;
        if (e < least || (e == least && which != 0xFFFFFFFFu && number < which)) {
            least = e;
            which = number;
        }
    }
    if (eq[0] && eq[1] && eq[2]) {
        // equal endpoints: one colour and black; a lane per (low end's moves),
        // the high end's follow
        const uint32_t d[3] = {lane % 3, lane / 3 % 3, lane / 9 % 3};
        bool ok = lane < 27;
        int c[3];
        uint32_t number = 0, scale = 1;
        for (uint32_t k = 0; k < 3; k++) {
            c[k] = E.e[0][k] + (int)d[k] - 1;
            const int h = c[k] - E.e[1][k] + 1;
            ok &= h >= 0 && h <= 2 && c[k] >= 0 && c[k] <= (k == 1 ? 63 : 31);
            number += scale * (d[k] + 27u * (uint32_t)max(h, 0));
            scale *= 3;
        }
        int p[3];
        expand565(pack565(c) & 0xFFFFu, p);
        const int black[3] = {0, 0, 0};
        uint32_t e = 0;
        for (uint32_t t = 0; t < 16; t++) {
            const uint32_t px = lane_value(B.own, t);
            e += min(colour_distance(px, p), colour_distance(px, black));
        }
        if (ok && number != 364 && (e < least || (e == least && which != 0xFFFFFFFFu && number < which))) {
            least = e;
            which = number;
        }
    }
    // the wave's smallest error, the lowest number on ties
    const uint32_t me = wave_min(which == 0xFFFFFFFFu ? 0xFFFFFFFFu : least);
    if (me == 0xFFFFFFFFu) return false;
    const uint32_t m = wave_min(which != 0xFFFFFFFFu && least == me ? which : 0xFFFFFFFFu);
    uint32_t r = m;
    for (int s = 0; s < 2; s++)
        for (int k = 0; k < 3; k++) {
            E.e[s][k] += (int)(r % 3) - 1;
            r /= 3;
        }
    best = me;
    return true;
}

__device__ inline WaveBlock wave_block(const uint8_t* px)
{
    const uint32_t lane = threadIdx.x & 63u;
    WaveBlock B;
    __builtin_memcpy(&B.own, px + 4 * (lane & 15u), 4);   // any alignment
    for (uint32_t j = 0; j < 4; j++) B.quad[j] = (uint32_t)__shfl((int)B.own, (int)(4 * (lane & 3u) + j));
    return B;
}

// Up to four lattice steps from E; true if any improved.
__device__ inline bool wave_polish(PolishLds& L, const WaveBlock& B, Ends& E, uint32_t& best, uint32_t max_iters,
                                   bool refit, uint32_t& steps)
{
    const uint32_t group = (threadIdx.x & 63u) >> 4;
    const uint32_t r = B.own & 255u, g = (B.own >> 8) & 255u, b = (B.own >> 16) & 255u;
    const int own_rg = (int)lane_value(row_sum(8 * r * r + 25 * g * g), 0);
    const int own_b = (int)lane_value(row_sum(b * b), 0);
    u32x4 texels = {0u, 0u, 0u, 0u};
    if (group == 0) texels = u32x4{bf2((float)r, 1.0f), bf2(1.0f, 1.0f), 0u, 0u};
    if (group == 1) texels = u32x4{bf2((float)g, (float)g), bf2((float)g, 1.0f), bf2(1.0f, 1.0f), 0u};
    if (group == 2) texels = u32x4{bf2((float)b, 1.0f), bf2(1.0f, 1.0f), 0u, 0u};
    bool moved = false;
    for (int it = 0; it < 4 && best; it++) {
        if (!wave_box_step(L, B, texels, own_rg, own_b, E, best)) break;
        moved = true;
        best = wave_refine(B, E, max_iters, refit, steps);
    }
    return moved;
}

// The output record of a block's endpoints.
__device__ inline u32x4 wave_record(const WaveBlock& B, const Ends& E, uint32_t best, uint32_t steps)
{
    const uint32_t ca = pack565(E.e[0]), cb = pack565(E.e[1]);
    uint32_t sel = own_selector(B, E.e[0], E.e[1]) << (2 * (threadIdx.x & 15u));
    sel |= dpp_of<0x128>(sel);
    sel |= dpp_of<0x124>(sel);
    sel |= dpp_of<0x122>(sel);
    sel |= dpp_of<0x121>(sel);
    return u32x4{max(ca, cb) | min(ca, cb) << 16, sel, best, steps};
}

constexpr uint32_t kPolishWaves = 4;

__global__ void __launch_bounds__(64 * kPolishWaves) polish_kernel(const uint8_t* __restrict__ rgba, uint32_t n,
                                                                   uint32_t per, uint32_t max_iters, uint32_t refit,
                                                                   uint32_t* __restrict__ out)
{
    __shared__ PolishLds lds[kPolishWaves];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63u;
    PolishLds& L = lds[wave];
    const uint64_t first = ((uint64_t)blockIdx.x * kPolishWaves + wave) * per;
    if (first >= n) return;
    const uint32_t m = (uint32_t)min((uint64_t)per, n - first);
    if (lane == 0) L.zero = u32x4{0u, 0u, 0u, 0u};
    __builtin_amdgcn_wave_barrier();
    // one block's state per lane; blocks of error zero have nothing to gain
    uint32_t* rec = out + 4 * (first + min(lane, m - 1));
    u32x4 mine;
    __builtin_memcpy(&mine, rec, 16);   // (no more than the output's own alignment is known)
    const uint64_t blocks = m == 64 ? ~0ull : (1ull << m) - 1ull;
    uint64_t todo = __ballot(mine.z != 0) & blocks;
    const uint32_t swapped = mine.w & kSwapped;
    mine.w &= ~kSwapped;
    while (todo) {
        const uint32_t k = (uint32_t)__builtin_ctzll(todo);
        todo &= todo - 1;
        const WaveBlock B = wave_block(rgba + (first + k) * 64);
        const uint32_t lohi = lane_value(mine.x, k), sw = lane_value(swapped, k);
        uint32_t best = lane_value(mine.z, k), steps = lane_value(mine.w, k);
        const uint32_t cc[2] = {sw ? lohi >> 16 : lohi & 0xFFFFu, sw ? lohi & 0xFFFFu : lohi >> 16};
        Ends E;
        for (int s = 0; s < 2; s++) {
            E.e[s][0] = (int)(cc[s] >> 11);
            E.e[s][1] = (int)((cc[s] >> 5) & 63u);
            E.e[s][2] = (int)(cc[s] & 31u);
        }
        if (wave_polish(L, B, E, best, max_iters, refit != 0, steps)) {
            const u32x4 q = wave_record(B, E, best, steps);
            if (lane == k) mine = q;
        }
    }
    if (lane < m) __builtin_memcpy(rec, &mine, 16);
}

// The whole refinement, one wavefront per block: for calls whose blocks would
// leave refine_kernel's one lane per block a wave or less per SIMD, where its
// time is that of the slowest block (4,096 blocks 3.68 ms with the polish in it,
// here 74 us).  Beyond kWaveBlocks blocks refine_kernel's lanes do more work per
// operation: 65,536 blocks, one lane per block / here, without the polish 455 /
// 510 us, of near-flat blocks with it 553 to 753 / 837, of a texture 702 / 677;
// 49,152 blocks 451 / 386, 515 / 631 (767 with the polish in it), 639 / 512.
constexpr uint32_t kWaveBlocks = 57344;

__global__ void __launch_bounds__(64 * kPolishWaves) refine_wave_kernel(const uint8_t* __restrict__ rgba, uint32_t n,
                                                                        const float* __restrict__ y,
                                                                        uint32_t max_iters, uint32_t starts,
                                                                        uint32_t* __restrict__ out)
{
    __shared__ PolishLds lds[kPolishWaves];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63u;
    PolishLds& L = lds[wave];
    const uint32_t b = blockIdx.x * kPolishWaves + wave;
    if (b >= n) return;
    if (lane == 0) L.zero = u32x4{0u, 0u, 0u, 0u};
    __builtin_amdgcn_wave_barrier();
    const WaveBlock B = wave_block(rgba + (size_t)b * 64);
    int px[16][3];
#pragma unroll
    for (int i = 0; i < 16; i++)
        for (int k = 0; k < 3; k++) px[i][k] = (int)((lane_value(B.own, (uint32_t)i) >> (8 * k)) & 255u);
    const bool refit = (starts & 8u) != 0;
    uint32_t best = 0xFFFFFFFFu, steps = 0;
    Ends keep = {{{0, 0, 0}, {0, 0, 0}}};
    for (uint32_t t = 0; t < 3; t++) {
        if (!(starts >> t & 1u)) continue;
        Ends E;
        if (t == 0) net_start(y + (size_t)b * 8, E.e);
        else if (t == 1) box_start(px, E.e);
        else pca_start(px, E.e);
        const uint32_t eb = wave_refine(B, E, max_iters, refit, steps);
        if (eb < best) {
            best = eb;
            keep = E;
        }
    }
    if (starts & 16u) wave_polish(L, B, keep, best, max_iters, refit, steps);
    const u32x4 q = wave_record(B, keep, best, steps);
    if (lane == 0) __builtin_memcpy(out + 4 * (size_t)b, &q, 16);
}

// Error of given DXT1 blocks (c0 | c1 << 16 per block) under the same decode.
__global__ void __launch_bounds__(256) block_error_kernel(const uint8_t* __restrict__ rgba, uint32_t n,
                                                          const uint32_t* __restrict__ ends, uint32_t stride,
                                                          uint32_t* __restrict__ err, uint32_t* __restrict__ sel)
{
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= n) return;
    int px[16][3];
    for (int i = 0; i < 16; i++)
        for (int k = 0; k < 3; k++) px[i][k] = rgba[(size_t)b * 64 + 4 * i + k];
    const uint32_t e = ends[(size_t)b * stride];
    uint32_t s;
    err[b] = dxt1_error(px, e & 0xFFFFu, e >> 16, &s);
    if (sel) sel[b] = s;
}

inline uint32_t grid1(uint64_t n, uint32_t tb) { return (uint32_t)((n + tb - 1) / tb); }

}  // namespace

extern "C" {

int crn2_mlp_features_device(const void* rgba, uint32_t n, float* feat, void* stream)
{
    if (!n) return CRN2_OK;
    if (!rgba || !feat) return CRN2_EINVAL;
    hipLaunchKernelGGL(mlp_features_kernel, dim3(grid1(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint8_t*>(rgba), n, feat);
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

int crn2_gemm_f32_device(uint32_t M, uint32_t N, uint32_t K, const float* A, int64_t sam, int64_t sak, const float* B,
                         int64_t sbk, int64_t sbn, float* C, int64_t ldc, int accumulate, int round_a, int round_b,
                         uint32_t ksplit, void* stream)
{
    if (!M || !N) return CRN2_OK;
    if (!A || !B || !C || !ksplit || ksplit > 1024) return CRN2_EINVAL;
    GemmArgs g{A, B, C, M, N, K, sam, sak, sbk, sbn, ldc, accumulate, round_a, round_b};
    hipLaunchKernelGGL(gemm_f32_kernel, dim3((N + 63) / 64, (M + 63) / 64, ksplit), dim3(256), 0,
                       static_cast<hipStream_t>(stream), g);
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

int crn2_mlp_bias_act_device(float* Z, float* A, const float* bias, uint32_t rows, uint32_t cols, int use_gelu,
                             void* stream)
{
    const uint64_t n = (uint64_t)rows * cols;
    if (!n) return CRN2_OK;
    hipLaunchKernelGGL(bias_act_kernel, dim3(grid1(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), Z, A,
                       bias, rows, cols, use_gelu);
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

int crn2_mlp_gelu_back_device(const float* dA, const float* Z, float* dZ, uint64_t n, void* stream)
{
    if (!n) return CRN2_OK;
    hipLaunchKernelGGL(gelu_back_kernel, dim3(grid1(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), dA, Z,
                       dZ, n);
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

int crn2_mlp_loss_device(const float* Y, const float* T, const float* labels, uint32_t rows, float* dY, float* loss,
                         void* stream)
{
    if (!rows) return CRN2_OK;
    hipLaunchKernelGGL(mlp_loss_kernel, dim3(grid1(rows, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), Y, T,
                       labels, rows, dY, loss);
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

uint64_t crn2_mlp_gradients_work(uint32_t rows) { return rows ? (uint64_t)grad_wgs(rows) * kPartial : 0; }

int crn2_mlp_gradients_device(const float* X, const float* T, const float* labels, uint32_t rows, const float* theta,
                              float* g, float* loss, float* work, uint64_t work_floats, void* stream)
{
    if (!theta || !g || !loss || (rows && (!X || !T || !work || work_floats < crn2_mlp_gradients_work(rows))))
        return CRN2_EINVAL;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint32_t wgs = rows ? grad_wgs(rows) : 0;
    if (rows) {
        // the LDS limit is a property of the kernel on each device: set it once per device
        static std::once_flag once[64];
        static bool ready[64];
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return CRN2_EHIP;
        std::call_once(once[dev], [&] {
            ready[dev] = hipFuncSetAttribute(reinterpret_cast<const void*>(&mlp_grad_kernel<32>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)sizeof(GradLds<32>)) == hipSuccess &&
                         hipFuncSetAttribute(reinterpret_cast<const void*>(&mlp_grad_kernel<64>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)sizeof(GradLds<64>)) == hipSuccess;
        });
        if (!ready[dev]) return CRN2_EHIP;
        if (grad_rows(rows) == 32)
            hipLaunchKernelGGL(mlp_grad_kernel<32>, dim3(wgs), dim3(256), sizeof(GradLds<32>), st, X, T, labels, rows,
                               theta, work);
        else
            hipLaunchKernelGGL(mlp_grad_kernel<64>, dim3(wgs), dim3(256), sizeof(GradLds<64>), st, X, T, labels, rows,
                               theta, work);
        if (hipGetLastError() != hipSuccess) return CRN2_EHIP;
    }
    hipLaunchKernelGGL(mlp_grad_reduce_kernel, dim3((kPartial + 63) / 64), dim3(256), 0, st, work, wgs, g, loss,
                       rows ? rows : 1u);
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

int crn2_adam_device(float* w, const float* g, float* m, float* v, uint32_t n, float lr, float b1, float b2, float eps,
                     uint32_t step, void* stream)
{
    if (!n) return CRN2_OK;
    const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
    hipLaunchKernelGGL(adam_kernel, dim3(grid1(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), w, g, m, v, n,
                       lr, b1, b2, eps, c1, c2);
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

int crn2_mlp_infer_device(const void* rgba, uint32_t n, const float* theta, float* y, void* stream)
{
    if (!n) return CRN2_OK;
    if (!rgba || !theta || !y) return CRN2_EINVAL;
    // the LDS limit is a property of the kernel on each device: set it once per device
    static bool attr[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return CRN2_EHIP;
    if (!attr[dev]) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&mlp_infer_kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kInferLds) != hipSuccess)
            return CRN2_EHIP;
        attr[dev] = true;
    }
    const uint32_t tiles = (n + 31) / 32;
    const uint32_t wgs = std::min<uint32_t>((tiles + kInferWaves - 1) / kInferWaves, 1024);
    hipLaunchKernelGGL(mlp_infer_kernel, dim3(wgs), dim3(256), kInferLds, static_cast<hipStream_t>(stream),
                       static_cast<const uint8_t*>(rgba), n, theta, y);
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

int crn2_dxt1_refine_device(const void* rgba, uint32_t n, const float* y, uint32_t max_iters, uint32_t starts,
                            uint32_t* out, void* stream)
{
    if (!n) return CRN2_OK;
    if (!rgba || !out || !(starts & 7u) || (starts & ~31u) || ((starts & 1u) && !y)) return CRN2_EINVAL;
    if (n <= kWaveBlocks) {
        hipLaunchKernelGGL(refine_wave_kernel, dim3(grid1(n, kPolishWaves)), dim3(64 * kPolishWaves), 0,
                           static_cast<hipStream_t>(stream), static_cast<const uint8_t*>(rgba), n, y, max_iters, starts,
                           out);
        return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
    }
    hipLaunchKernelGGL(refine_kernel, dim3(grid1(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint8_t*>(rgba), n, y, max_iters, starts, out);
    if (hipGetLastError() != hipSuccess) return CRN2_EHIP;
    if (starts & 16u) {
        // blocks per wave: one until the waves fill the GPU many times over
        const uint32_t per = std::min<uint32_t>(64, std::max<uint32_t>(1, n >> 16));
        hipLaunchKernelGGL(polish_kernel, dim3(grid1(n, per * kPolishWaves)), dim3(64 * kPolishWaves), 0,
                           static_cast<hipStream_t>(stream), static_cast<const uint8_t*>(rgba), n, per, max_iters,
                           (starts >> 3) & 1u, out);
        if (hipGetLastError() != hipSuccess) return CRN2_EHIP;
    }
    return CRN2_OK;
}

int crn2_dxt1_block_error_device(const void* rgba, uint32_t n, const uint32_t* endpoints, uint32_t stride_u32,
                                 uint32_t* err, uint32_t* selectors, void* stream)
{
    if (!n) return CRN2_OK;
    if (!rgba || !endpoints || !err || !stride_u32) return CRN2_EINVAL;
    hipLaunchKernelGGL(block_error_kernel, dim3(grid1(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint8_t*>(rgba), n, endpoints, stride_u32, err, selectors);
    return hipGetLastError() == hipSuccess ? CRN2_OK : CRN2_EHIP;
}

}  // extern "C"
