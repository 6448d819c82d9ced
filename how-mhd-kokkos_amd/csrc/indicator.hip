// Learned smoothness indicator: inference, training (forward + backward with
// the weight gradients on bf16 MFMA, FP32 accumulation) and Adam, behind the
// C-ABI of include/howmhd_mlp.h.
//
// Training numerics (the CPU check in tests/ follows the same definitions):
//   forward  x, W1, W2 rounded to bf16; z1 = x W1^T + b1 (FP32 accumulate);
//            a1 = bf16(relu(z1)); z2 = a1 W2^T + b2; a2 = bf16(relu(z2));
//            z3 = b3 + sum_j a2_j * bf16(w3_j) in FP32, j = 0..31
//   loss     w * (softplus(z3) - y z3), w = pos_weight for y = 1 else 1
//   backward dz3 = w (sigmoid(z3) - y) * scale (FP32)
//            dw3 = sum_i dz3 a2, db3 = sum_i dz3 (FP32)
//            dz2 = bf16(dz3 * bf16(w3) where a2 != 0); dW2 = dz2^T a1; db2 = sum_i dz2
//            dz1 = bf16((dz2 W2) where a1 != 0);       dW1 = dz1^T x;  db1 = sum_i dz1
#include "howmhd_mlp.h"
#include "mlp.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

using namespace howmhd;

namespace {

// Both kernels give a wavefront tiles of 16 samples and keep a tile in
// registers from the features to the logit (and back).  With q = lane / 16,
// every layer is a v_mfma_f32_16x16x16_bf16 product over two k-steps of 16,
// in one of two orientations:
//   unit-major    D = W X^T: the lane holds sample lane % 16, units 4q..4q+3
//                 of each 16-unit tile.  This is the next layer's operand as
//                 it lies (k = 4q + v), so layers chain without moving data.
//   sample-major  D = X W^T (the operands exchanged): the lane holds unit
//                 lane % 16, samples 4q..4q+3: the operand layout of a
//                 contraction over samples, which the weight gradients are.
// The output layer's w3 fills all 16 rows of its operand, so that every lane
// receives the logit of its sample.

typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bf16x4 pack4(f32x4 v) {
    bf16x4 r;
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = (short)f2bf(v[k]);
    return r;
}
__device__ __forceinline__ bf16x4 relu4(f32x4 z) {
#pragma unroll
    for (int k = 0; k < 4; ++k) z[k] = z[k] > 0.f ? z[k] : 0.f;
    return pack4(z);
}

// Four floats at P[j..j+3] that need only 4-byte alignment.
__device__ __forceinline__ f32x4 load4(const float* P) { return *reinterpret_cast<const f32x4u*>(P); }

// This lane's part of the network: operand fragments of the forward products
// (rows of W: unit 16u + lane % 16, k = 16s + 4q + v), unit-major biases and
// the output layer.
struct Net {
    bf16x4 W1[2][2], W2[2][2], w3[2];  // [k-step s][unit tile u]; w3[s]
    f32x4 b1[2], b2[2];                // unit-major accumulator rows 16u + 4q + v
    float b3;
};

__device__ __forceinline__ void load_net(const float* P, Net& N) {
    const int l = threadIdx.x & 63, r16 = l % 16, q4 = 4 * (l / 16);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const float* w1 = P + MLP_OFF_W1 + (16 * u + r16) * MLP_IN;
        N.W1[0][u] = pack4(load4(w1 + q4));
        f32x4 t = {0.f, 0.f, 0.f, 0.f};
        if (q4 == 0) { t[0] = w1[16]; t[1] = w1[17]; }  // features 16, 17; the rest of k-step 1 is 0
        N.W1[1][u] = pack4(t);
#pragma unroll
        for (int s = 0; s < 2; ++s) N.W2[s][u] = pack4(load4(P + MLP_OFF_W2 + (16 * u + r16) * MLP_H + 16 * s + q4));
        N.w3[u] = pack4(load4(P + MLP_OFF_W3 + 16 * u + q4));
        N.b1[u] = load4(P + MLP_OFF_B1 + 16 * u + q4);
        N.b2[u] = load4(P + MLP_OFF_B2 + 16 * u + q4);
    }
    N.b3 = P[MLP_OFF_B3];
}

// Features of sample i as the lane's k-slots of the first layer: 4q..4q+3 and
// (q = 0) 16, 17; zeros for a sample beyond the last.  X rows are 72 B, so the
// 16-byte loads need no more than the 4-byte alignment that X has.
__device__ __forceinline__ void load_x(const float* X, int64_t i, int64_t n, f32x4& x0, f32x4& x1) {
    const int q4 = 4 * ((threadIdx.x & 63) / 16);
    x0 = f32x4{0.f, 0.f, 0.f, 0.f};
    x1 = f32x4{0.f, 0.f, 0.f, 0.f};
    if (i < n) {
        const float* x = X + i * MLP_IN;
        x0 = load4(x + q4);
        if (q4 == 0) {
            const f32x2u t = *reinterpret_cast<const f32x2u*>(x + 16);
            x1[0] = t[0];
            x1[1] = t[1];
        }
    }
}

// One layer, unit-major: D[u] = bias + W h^T, h[s] the k-step operands.
__device__ __forceinline__ void layer_u(const bf16x4 (*W)[2], const f32x4* bias, const bf16x4* h, f32x4* z) {
#pragma unroll
    for (int u = 0; u < 2; ++u) z[u] = mfma16(W[1][u], h[1], mfma16(W[0][u], h[0], bias[u]));
}

// Logits.  Bound: the 76 B a sample moves.  A wavefront loads the weights
// once and strides over groups of four tiles, whose loads are in flight
// together: 2e6 samples take 29 us (5.2 TB/s, a device copy's rate); with the
// weights built for every 64 samples and the activations passed through LDS
// they took 99 us.  At most INFER_BLOCKS blocks; 1,024 to 4,096 time the same.
constexpr int INFER_TILES = 4;
constexpr int64_t INFER_BLOCKS = 2048;
__global__ __launch_bounds__(256) void k_mlp_infer(const float* X, int64_t n, const float* P, float* logits) {
    const int l = threadIdx.x & 63, r16 = l % 16, q = l / 16;
    const int64_t ngroup = (n + 63) / 64, stride = (int64_t)gridDim.x * 4;
    Net N;
    load_net(P, N);
    for (int64_t gidx = (int64_t)blockIdx.x * 4 + threadIdx.x / 64; gidx < ngroup; gidx += stride) {
        const int64_t i0 = gidx * 64;
        f32x4 x0[INFER_TILES], x1[INFER_TILES];
#pragma unroll
        for (int t = 0; t < INFER_TILES; ++t) load_x(X, i0 + 16 * t + r16, n, x0[t], x1[t]);
        float out = 0.f;
#pragma unroll
        for (int t = 0; t < INFER_TILES; ++t) {
            bf16x4 h[2] = {pack4(x0[t]), pack4(x1[t])};
            f32x4 z[2];
            layer_u(N.W1, N.b1, h, z);
            h[0] = relu4(z[0]);
            h[1] = relu4(z[1]);
            layer_u(N.W2, N.b2, h, z);
            h[0] = relu4(z[0]);
            h[1] = relu4(z[1]);
            f32x4 o = {N.b3, N.b3, N.b3, N.b3};
            o = mfma16(N.w3[1], h[1], mfma16(N.w3[0], h[0], o));
            out = (q == t) ? o[0] : out;
        }
        if (i0 + l < n) logits[i0 + l] = out;
    }
}

// Gradient.  A wavefront strides over tiles and keeps its part of the
// gradient in registers (the weight gradients as MFMA accumulators, db1 as
// the product with a feature 18 that is 1); the block's wavefronts meet in
// LDS and every parameter gets one atomic per block.  Bound: small batches by
// those atomics (one address takes them one after the other) and the latency
// of a tile's chain, large ones by the vector instructions of a tile.  One
// atomic per parameter and wavefront of 64 samples took 93.5 us for 1,024
// tiles (16,384 samples) and 7.7 ms for 2e6 samples; this takes 9.2 us and
// 137 us.  8 wavefronts a block: 4 or 16 take 13.1 or 21.9 us at 16,384
// samples; 2 tiles per wavefront at least 9.5 us; 512 blocks at most 143 us at
// 2e6 (only 256 are resident at 188 registers).
constexpr int GRAD_WAVES = 8;
constexpr int64_t GRAD_BLOCKS = 256;

__global__ __launch_bounds__(64 * GRAD_WAVES) void k_mlp_grad(const float* X, const float* Y, int64_t n,
                                                              const float* P, float pos_weight, float scale, float* G,
                                                              float* loss) {
    __shared__ float parts[GRAD_WAVES][MLP_NPARAM + 1];  // per wavefront: the gradient, then the loss
    const int l = threadIdx.x & 63, r16 = l % 16, q = l / 16, q4 = 4 * q;
    Net N;
    load_net(P, N);
    // sample-major forms: biases and w3 of unit 16u + lane % 16, w3 of units
    // 16u + 4q + v, and W2 as the right operand of dz1 = dz2 W2
    // (k = unit of layer 2, column = unit 16u + lane % 16 of layer 1)
    float b1s[2], b2s[2], w3s[2];
    f32x4 w3u[2];
    bf16x4 W2b[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        b1s[u] = P[MLP_OFF_B1 + 16 * u + r16];
        b2s[u] = P[MLP_OFF_B2 + 16 * u + r16];
        w3s[u] = bf2f(f2bf(P[MLP_OFF_W3 + 16 * u + r16]));
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            w3u[u][v] = bf2f((uint16_t)N.w3[u][v]);
#pragma unroll
            for (int s = 0; s < 2; ++s)
                W2b[s][u][v] = (short)f2bf(P[MLP_OFF_W2 + (16 * s + q4 + v) * MLP_H + 16 * u + r16]);
        }
    }
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 gW2[2][2] = {{zero, zero}, {zero, zero}}, gW1[2][2] = {{zero, zero}, {zero, zero}};
    float gb2[2] = {0.f, 0.f}, gw3[2] = {0.f, 0.f}, gb3 = 0.f, gl = 0.f;

    const int64_t ntile = (n + 15) / 16, stride = (int64_t)gridDim.x * GRAD_WAVES;
    for (int64_t t = (int64_t)blockIdx.x * GRAD_WAVES + threadIdx.x / 64; t < ntile; t += stride) {
        const int64_t i0 = 16 * t, i = i0 + r16;
        f32x4 x0, x1;
        load_x(X, i, n, x0, x1);
        // features of samples 4q..4q+3 (rows of the dW1 product): feature
        // lane % 16, and 16 + lane % 16 with the 1 of db1 at 18
        f32x4 xs[2] = {zero, zero};
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int64_t k = i0 + q4 + v;
            if (k < n) {
                xs[0][v] = X[k * MLP_IN + r16];
                if (r16 < 2) xs[1][v] = X[k * MLP_IN + 16 + r16];
                else if (r16 == 2) xs[1][v] = 1.f;
            }
        }
        const bool valid = i < n;
        const float yv = valid ? Y[i] : 0.f;

        // ---- forward, both orientations
        const bf16x4 x[2] = {pack4(x0), pack4(x1)};
        f32x4 z[2];
        bf16x4 a1[2], a1s[2], a2[2], a2s[2];
        layer_u(N.W1, N.b1, x, z);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            a1[u] = relu4(z[u]);
            const f32x4 b = {b1s[u], b1s[u], b1s[u], b1s[u]};
            a1s[u] = relu4(mfma16(x[1], N.W1[1][u], mfma16(x[0], N.W1[0][u], b)));
        }
        layer_u(N.W2, N.b2, a1, z);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            a2[u] = relu4(z[u]);
            const f32x4 b = {b2s[u], b2s[u], b2s[u], b2s[u]};
            a2s[u] = relu4(mfma16(a1[1], N.W2[1][u], mfma16(a1[0], N.W2[0][u], b)));
        }
        f32x4 o = {N.b3, N.b3, N.b3, N.b3};
        o = mfma16(N.w3[1], a2[1], mfma16(N.w3[0], a2[0], o));
        const float z3 = o[0];

        // ---- loss and output layer
        const float wgt = (yv > 0.5f) ? pos_weight : 1.f;
        const float p = 1.f / (1.f + expf(-z3));
        const float dz3 = valid ? wgt * (p - yv) * scale : 0.f;
        // (the four quarters of the wavefront hold the same samples)
        gl += valid ? wgt * (fmaxf(z3, 0.f) + log1pf(expf(-fabsf(z3))) - yv * z3) * scale : 0.f;
        gb3 += dz3;
        float dz3s[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) dz3s[v] = __shfl(dz3, q4 + v, 64);

        // ---- dz2 = dz3 w3 where a2 != 0
        bf16x4 d2[2], d2s[2], d1s[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                d2[u][v] = a2[u][v] != 0 ? (short)f2bf(dz3 * w3u[u][v]) : (short)0;
                d2s[u][v] = a2s[u][v] != 0 ? (short)f2bf(dz3s[v] * w3s[u]) : (short)0;
                gw3[u] += dz3s[v] * bf2f((uint16_t)a2s[u][v]);
                gb2[u] += bf2f((uint16_t)d2s[u][v]);
            }
        // ---- dz1 = dz2 W2 where a1 != 0
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const f32x4 c = mfma16(d2[1], W2b[1][u], mfma16(d2[0], W2b[0][u], zero));
#pragma unroll
            for (int v = 0; v < 4; ++v) d1s[u][v] = a1s[u][v] != 0 ? (short)f2bf(c[v]) : (short)0;
        }
        // ---- dW2 += dz2^T a1, dW1 += dz1^T x
        const bf16x4 xb[2] = {pack4(xs[0]), pack4(xs[1])};
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                gW2[m][u] = mfma16(d2s[m], a1s[u], gW2[m][u]);
                gW1[m][u] = mfma16(d1s[m], xb[u], gW1[m][u]);
            }
    }

    // ---- the block's sum: each wavefront's part in LDS, then added in order
    auto quarters = [](float x) {  // sum over the four lanes with the same lane % 16
        x += __shfl_xor(x, 16, 64);
        return x + __shfl_xor(x, 32, 64);
    };
    float* part = parts[threadIdx.x / 64];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 16 * m + q4 + v, col = 16 * u + r16;
                part[MLP_OFF_W2 + row * MLP_H + col] = gW2[m][u][v];
                if (col < MLP_IN) part[MLP_OFF_W1 + row * MLP_IN + col] = gW1[m][u][v];
                else if (col == MLP_IN) part[MLP_OFF_B1 + row] = gW1[m][u][v];
            }
        const float sb = quarters(gb2[m]), sw = quarters(gw3[m]);
        if (q == 0) {
            part[MLP_OFF_B2 + 16 * m + r16] = sb;
            part[MLP_OFF_W3 + 16 * m + r16] = sw;
        }
    }
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) {  // over the 16 samples of a quarter
        gb3 += __shfl_xor(gb3, off, 64);
        gl += __shfl_xor(gl, off, 64);
    }
    if (l == 0) {
        part[MLP_OFF_B3] = gb3;
        part[MLP_NPARAM] = gl;
    }
    __syncthreads();
    for (int j = threadIdx.x; j < MLP_NPARAM + 1; j += 64 * GRAD_WAVES) {
        float sum = parts[0][j];
#pragma unroll
        for (int w = 1; w < GRAD_WAVES; ++w) sum += parts[w][j];
        atomicAdd(j < MLP_NPARAM ? &G[j] : loss, sum);
    }
}

__global__ void k_mlp_adam(float* P, float* M, float* V, const float* G, float lr, float b1, float b2, float eps,
                           float c1, float c2) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= MLP_NPARAM) return;
    const float g = G[j];
    const float m = b1 * M[j] + (1.f - b1) * g;
    const float v = b2 * V[j] + (1.f - b2) * g * g;
    M[j] = m;
    V[j] = v;
    P[j] -= lr * (m / c1) / (sqrtf(v / c2) + eps);
}

}  // namespace

extern "C" {

int howmhd_mlp_infer(const float* X, int64_t n, const float* params, float* logits, void* stream) {
    if (n <= 0) return HOWMHD_OK;
    if (!X || !params || !logits) return HOWMHD_EINVAL;
    // at most 8 blocks per CU (all resident), so that larger sets amortise
    // the weights over several groups per wavefront
    const unsigned nb = (unsigned)std::min<int64_t>((n + 255) / 256, INFER_BLOCKS);
    hipLaunchKernelGGL(k_mlp_infer, dim3(nb), dim3(256), 0, (hipStream_t)stream, X, n, params, logits);
    return hipGetLastError() == hipSuccess ? HOWMHD_OK : HOWMHD_EHIP;
}

int howmhd_mlp_grad(const float* X, const float* y, int64_t n, const float* params, float pos_weight,
                    float scale, float* grad, float* loss, void* stream) {
    if (n <= 0) return HOWMHD_OK;
    if (!X || !y || !params || !grad || !loss) return HOWMHD_EINVAL;
    const int64_t per_block = 16 * GRAD_WAVES;
    const unsigned nb = (unsigned)std::min<int64_t>((n + per_block - 1) / per_block, GRAD_BLOCKS);
    hipLaunchKernelGGL(k_mlp_grad, dim3(nb), dim3(64 * GRAD_WAVES), 0, (hipStream_t)stream, X, y, n, params, pos_weight, scale,
                       grad, loss);
    return hipGetLastError() == hipSuccess ? HOWMHD_OK : HOWMHD_EHIP;
}

int howmhd_mlp_adam(float* params, float* m, float* v, const float* grad, int64_t t, float lr, float beta1,
                    float beta2, float eps, void* stream) {
    if (!params || !m || !v || !grad || t < 1) return HOWMHD_EINVAL;
    const float c1 = 1.f - powf(beta1, (float)t);
    const float c2 = 1.f - powf(beta2, (float)t);
    hipLaunchKernelGGL(k_mlp_adam, dim3((MLP_NPARAM + 255) / 256), dim3(256), 0, (hipStream_t)stream, params, m, v,
                       grad, lr, beta1, beta2, eps, c1, c2);
    return hipGetLastError() == hipSuccess ? HOWMHD_OK : HOWMHD_EHIP;
}

}  // extern "C"
