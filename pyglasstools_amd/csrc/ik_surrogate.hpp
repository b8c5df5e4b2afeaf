// ik_surrogate.hpp -- the learned bond-integral surrogate (gfx950).
// Included by ik_kernels.hpp.
//
// A tanh MLP 5 -> 64 -> 64 -> 64 -> 1 maps a bond seen from a grid point,
//   x = (a_x, a_y, b_x, b_y, r_cg),  a = (r_i - x) / r_cg,  b = (r_j - x) / r_cg,
// to the unnormalised Octic line integral w = sum_k w_k shape(|a + s_k (b - a)|^2)
// of the 5-node rule (2D).  Training runs in FP32 on the kernels below
// (dense forward, backward, mean-squared loss, Adam); inference runs in BF16
// on the matrix cores (v_mfma_f32_16x16x16_bf16) with FP32 accumulation.
//
// The field form with the surrogate enumerates the (grid point, bond) pairs
// of a frame into a pair buffer (k_pair_count, a scan, k_pair_write), infers
// w for every pair (k_mlp_infer), keeps it where the calibrated error bound
// of the pair's class is within the tolerance and recomputes it by the
// quadrature elsewhere (k_pair_finalize), and sums c' w b' (x) b' per grid
// point in pair order in FP64 (k_pair_reduce).
#pragma once
#include <hip/hip_runtime.h>

#include "ik_device.hpp"

namespace pgt {

// parameter layout (FP32): W1[5][64] b1[64] W2[64][64] b2[64] W3[64][64] b3[64] W4[64] b4
constexpr int kMlpIn = 5;
constexpr int kMlpInPad = 8;  // floats per input row in memory
constexpr int kMlpW = 64;
constexpr int kOffW1 = 0, kOffB1 = kOffW1 + kMlpIn * kMlpW, kOffW2 = kOffB1 + kMlpW, kOffB2 = kOffW2 + kMlpW * kMlpW,
              kOffW3 = kOffB2 + kMlpW, kOffB3 = kOffW3 + kMlpW * kMlpW, kOffW4 = kOffB3 + kMlpW,
              kOffB4 = kOffW4 + kMlpW, kMlpNParam = kOffB4 + 1;

// ------------------------------------------------------------------------
// FP32 training kernels (row-major activations, one sample per row)
// ------------------------------------------------------------------------

// Y[s][o] = act(b[o] + sum_k X[s][k] W[k][o]); X rows have stride ldx.  The
// layer sizes are template arguments, so a thread's K loads of X and of W
// issue together instead of one per step of a loop of unknown length.
template <int K, int N>
__global__ __launch_bounds__(256) void k_dense_fwd(int64_t n, const float *__restrict__ X, int ldx,
                                                   const float *__restrict__ W, const float *__restrict__ b,
                                                   bool tanh_act, float *__restrict__ Y)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n * N) return;
    const int64_t s = idx / N;
    const int o = (int)(idx % N);
    float x[K];
#pragma unroll
    for (int k = 0; k < K; ++k) x[k] = X[s * ldx + k];
    float acc = b[o];
#pragma unroll
    for (int k = 0; k < K; ++k) acc = fmaf(x[k], W[k * N + o], acc);
    Y[idx] = tanh_act ? tanhf(acc) : acc;
}

// Gradient of the mean-squared loss in one launch.  A workgroup takes chunks
// of C samples (chunk c, c + gridDim.x, ...) through the forward pass and
// back with every activation and error in LDS, and keeps its share of all
// weight gradients in registers; it then stores them, its bias gradients and
// its loss as row blockIdx.x of `part` (k_grad_sum adds the rows in order).
// As seventeen launches, one per layer and direction, the step of 1,024
// samples was bound by the launches and their tails: 65 us of kernels; this
// takes 9 us, the sum of the rows 3.4.
//
// The products run on the matrix cores in FP32 (v_mfma_f32_16x16x4_f32):
// wave w computes columns 16 w .. 16 w + 15.  Lane l = 16 q + c holds
// A[c][k] and B[k][c] of a step's four k, one per q, and D[4 q + r][c]; a
// product's k may come in any order, so that of step t is t + (K / 4) q, which
// makes a lane's A values neighbours.  The row strides (66 for activations and
// errors, 65 for weights) put the 64 lanes' words on distinct LDS banks.
constexpr int kGradMaxRows = 256;                   // workgroups
constexpr int kGradRow = (kMlpNParam + 3) / 4 * 4;  // floats of a row: the parameters' gradients, then
                                                    // (8-byte aligned, in the last two) the loss sum
static_assert(kGradRow >= ((kMlpNParam + 1) & ~1) + 2, "room for the loss");

// Samples of a chunk: 16 spread a batch over more CUs (64 workgroups for 1,024
// samples: 9.4 us a launch; 32 samples each on 32 workgroups, with the bias sums
// in one wavefront, 16.9), and would up to 4,096 samples, but only up to 1,177
// do a row for every 16 fit the workspace that callers allocate.
inline int grad_chunk(int64_t n) { return n <= 1024 ? 16 : 32; }
inline int grad_rows(int64_t n)
{
    const int64_t c = (n + grad_chunk(n) - 1) / grad_chunk(n);
    return (int)(c < kGradMaxRows ? c : kGradMaxRows);
}

template <int C>
__global__ __launch_bounds__(256) void k_mlp_grad(int64_t n, const float *__restrict__ P, const float *__restrict__ X,
                                                  const float *__restrict__ T, float *__restrict__ part)
{
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int W = kMlpW, AS = 66, WS = 65, NT = C / 16, KQ = C / 4;  // row tiles, samples per q
    __shared__ float s_w1[kMlpInPad][WS];  // rows past the inputs are zero
    __shared__ float s_w2[W][WS], s_w3[W][WS], s_w4[W], s_b[3][W];
    __shared__ float s_x[C][kMlpInPad + 2], s_h[3][C][AS], s_z[2][C][AS], s_dy[C];
    __shared__ double s_loss[4];
    __shared__ float s_gb4[4];
    const int t = threadIdx.x, w = t >> 6, l = t & 63, q = l >> 4, c = l & 15;
    const int col = 16 * w + c;
    {
        float v2[W * W / 256], v3[W * W / 256];  // all loads in flight together
#pragma unroll
        for (int k = 0; k < W * W / 256; ++k) {
            v2[k] = P[kOffW2 + 256 * k + t];
            v3[k] = P[kOffW3 + 256 * k + t];
        }
        for (int k = t; k < kMlpInPad * W; k += 256) s_w1[k / W][k % W] = k < kMlpIn * W ? P[kOffW1 + k] : 0.0f;
#pragma unroll
        for (int k = 0; k < W * W / 256; ++k) {
            s_w2[4 * k + w][l] = v2[k];
            s_w3[4 * k + w][l] = v3[k];
        }
    }
    if (t < W) {
        s_w4[t] = P[kOffW4 + t];
        s_b[0][t] = P[kOffB1 + t];
        s_b[1][t] = P[kOffB2 + t];
        s_b[2][t] = P[kOffB3 + t];
    }
    const float b4 = P[kOffB4];

    f32x4 g1{}, g2[4], g3[4];  // weight gradients: rows 16 i + 4 q + r of column col
#pragma unroll
    for (int i = 0; i < 4; ++i) g2[i] = g3[i] = f32x4{};
    float gw4 = 0.0f, gb[3] = {0.0f, 0.0f, 0.0f};  // of unit col
    float gb4 = 0.0f;   // of this thread's sample
    double loss = 0.0;

    // D = A (C x 64 activations or errors) B (64 x 64) for the wave's columns
    auto product = [&](const float (&A)[C][AS], auto bval, f32x4 (&d)[NT]) {
        float b[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) b[k] = bval(16 * q + k);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            d[i] = f32x4{};
            float a[16];
#pragma unroll
            for (int k = 0; k < 16; k += 2) {
                const float2 v = *reinterpret_cast<const float2 *>(&A[16 * i + c][16 * q + k]);
                a[k] = v.x;
                a[k + 1] = v.y;
            }
#pragma unroll
            for (int k = 0; k < 16; ++k) d[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[k], b[k], d[i], 0, 0, 0);
        }
    };
    // sum over the chunk's samples from the lane's KQ of them
    auto over_samples = [&](float v) {
        v += __shfl_xor(v, 16, 64);
        return v + __shfl_xor(v, 32, 64);
    };
    // G += A^T Z over the chunk's samples, and b += the sum of Z
    auto outer = [&](const float (&A)[C][AS], const float (&Z)[C][AS], f32x4 (&g)[4], float &b) {
        float z[KQ], v = 0.0f;
#pragma unroll
        for (int k = 0; k < KQ; ++k) {
            z[k] = Z[KQ * q + k][col];
            v += z[k];
        }
        b += over_samples(v);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int k = 0; k < KQ; ++k)
                g[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[KQ * q + k][16 * i + c], z[k], g[i], 0, 0, 0);
    };
    // the hidden layer's output from its pre-activations
    auto activate = [&](const f32x4 (&d)[NT], int layer) {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) s_h[layer][16 * i + 4 * q + r][col] = tanhf(d[i][r] + s_b[layer][col]);
    };
    // the error at a hidden layer's pre-activations
    auto error = [&](const f32x4 (&d)[NT], int layer, float (&Z)[C][AS]) {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float h = s_h[layer][16 * i + 4 * q + r][col];
                Z[16 * i + 4 * q + r][col] = d[i][r] * (1.0f - h * h);
            }
    };
    for (int64_t s0 = (int64_t)blockIdx.x * C; s0 < n; s0 += (int64_t)gridDim.x * C) {
        if (t < 8 * C) {
            const int r = t >> 3, k = t & 7;
            s_x[r][k] = s0 + r < n && k < kMlpIn ? X[(s0 + r) * kMlpInPad + k] : 0.0f;
        }
        __syncthreads();
        f32x4 d[NT];
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            d[i] = f32x4{};
#pragma unroll
            for (int k = 0; k < 2; ++k)
                d[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(s_x[16 * i + c][2 * q + k], s_w1[2 * q + k][col], d[i], 0, 0,
                                                            0);
        }
        activate(d, 0);
        __syncthreads();
        product(s_h[0], [&](int k) { return s_w2[k][col]; }, d);
        activate(d, 1);
        __syncthreads();
        product(s_h[1], [&](int k) { return s_w3[k][col]; }, d);
        activate(d, 2);
        __syncthreads();
        if (t < 8 * C) {  // the output and its error, eight threads per sample
            const int r = t >> 3, k0 = (t & 7) * 8;
            float y = 0.0f;
#pragma unroll
            for (int k = 0; k < 8; ++k) y = fmaf(s_h[2][r][k0 + k], s_w4[k0 + k], y);
#pragma unroll
            for (int off = 1; off < 8; off <<= 1) y += __shfl_xor(y, off, 64);
            if ((t & 7) == 0 && s0 + r < n) {
                const float e = y + b4 - T[s0 + r];
                const float dy = 2.0f * e / (float)n;
                s_dy[r] = dy;
                gb4 += dy;
                loss += (double)e * e;
            } else if ((t & 7) == 0) {
                s_dy[r] = 0.0f;
            }
        }
        __syncthreads();
        {
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < KQ; ++k) {
                const int r = KQ * q + k;
                const float h = s_h[2][r][col], dy = s_dy[r];
                v = fmaf(h, dy, v);
                s_z[0][r][col] = dy * s_w4[col] * (1.0f - h * h);
            }
            gw4 += over_samples(v);
        }
        __syncthreads();
        outer(s_h[1], s_z[0], g3, gb[2]);
        product(s_z[0], [&](int k) { return s_w3[col][k]; }, d);
        error(d, 1, s_z[1]);
        __syncthreads();
        outer(s_h[0], s_z[1], g2, gb[1]);
        product(s_z[1], [&](int k) { return s_w2[col][k]; }, d);
        error(d, 0, s_z[0]);
        __syncthreads();
        {
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < KQ; ++k) {
                const float z = s_z[0][KQ * q + k][col];
                v += z;
                g1 = __builtin_amdgcn_mfma_f32_16x16x4f32(c < kMlpIn ? s_x[KQ * q + k][c] : 0.0f, z, g1, 0, 0, 0);
            }
            gb[0] += over_samples(v);
        }
        __syncthreads();
    }

    // the samples' threads: a fixed butterfly, then the four wavefronts in order
#pragma unroll
    for (int off = 8; off < 64; off <<= 1) {
        gb4 += __shfl_xor(gb4, off, 64);
        loss += __shfl_xor(loss, off, 64);
    }
    if (l == 0) {
        s_gb4[w] = gb4;
        s_loss[w] = loss;
    }
    __syncthreads();
    float *out = part + (size_t)blockIdx.x * kGradRow;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (4 * q + r < kMlpIn) out[kOffW1 + (4 * q + r) * W + col] = g1[r];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            out[kOffW2 + (16 * i + 4 * q + r) * W + col] = g2[i][r];
            out[kOffW3 + (16 * i + 4 * q + r) * W + col] = g3[i][r];
        }
    }
    if (q == 0) {
        out[kOffB1 + col] = gb[0];
        out[kOffB2 + col] = gb[1];
        out[kOffB3 + col] = gb[2];
        out[kOffW4 + col] = gw4;
    }
    if (t == 0) {
        out[kOffB4] = s_gb4[0] + s_gb4[1] + s_gb4[2] + s_gb4[3];
        *reinterpret_cast<double *>(out + kGradRow - 2) = s_loss[0] + s_loss[1] + s_loss[2] + s_loss[3];
    }
}

// Sum of the values at p of rows r0 .. r1 - 1, in order.  16 loads are in
// flight together: with eight, and a loss sum that waited for each of its
// loads, k_grad_sum took 5.6 us for 64 rows and now takes 3.4; a step of 6,290
// samples (197 rows) 31.6 -> 23.4 us, of 7,940 35.4 -> 23.0.
template <typename T>
__device__ __forceinline__ T sum_rows(const float *__restrict__ p, int r0, int r1)
{
    constexpr int NB = 16;
    T s = T(0);
    for (int r = r0; r < r1; r += NB) {
        T x[NB];
#pragma unroll
        for (int u = 0; u < NB; ++u) x[u] = *reinterpret_cast<const T *>(p + (size_t)min(r + u, r1 - 1) * kGradRow);
#pragma unroll
        for (int u = 0; u < NB; ++u) s += r + u < r1 ? x[u] : T(0);
    }
    return s;
}

// grad = the sum of the rows of part, loss = the sum of their losses / n, each
// as four sums of consecutive rows added in order (64 parameters a workgroup).
__global__ __launch_bounds__(256) void k_grad_sum(int rows, const float *__restrict__ part, int64_t n,
                                                  float *__restrict__ grad, float *__restrict__ loss)
{
    __shared__ double sh[4][64];
    const int o = threadIdx.x & 63, u = threadIdx.x >> 6;
    const int k = blockIdx.x * 64 + o;
    const int r0 = rows * u / 4, r1 = rows * (u + 1) / 4;
    double v = 0.0;
    if (k < kMlpNParam) v = sum_rows<float>(part + k, r0, r1);
    else if (k == kMlpNParam) v = sum_rows<double>(part + kGradRow - 2, r0, r1);
    sh[u][o] = v;
    __syncthreads();
    if (u) return;
    if (k < kMlpNParam) grad[k] = (float)sh[0][o] + (float)sh[1][o] + (float)sh[2][o] + (float)sh[3][o];
    else if (k == kMlpNParam) loss[0] = (float)((sh[0][o] + sh[1][o] + sh[2][o] + sh[3][o]) / (double)n);
}

// Adam (Kingma & Ba 2015), bias-corrected, on np parameters.
__global__ void k_adam(int np, float *__restrict__ p, float *__restrict__ m, float *__restrict__ v,
                       const float *__restrict__ g, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ------------------------------------------------------------------------
// BF16 inference on the matrix cores
// ------------------------------------------------------------------------
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16 bits, round to nearest even (finite inputs).
__device__ __forceinline__ short to_bf16(float x)
{
    const unsigned u = __float_as_uint(x);
    return (short)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

// One wavefront evaluates 16 samples per step with v_mfma_f32_16x16x16_bf16.
// Every layer is computed transposed, D = W^T (out x in) * H^T (in x 16):
// lane l holds A[l % 16][4 (l / 16) + r] (weights), B[4 (l / 16) + r][l % 16]
// (activations) and D[4 (l / 16) + r][l % 16] (r = 0..3), so the D tile T of
// one layer, after bias and tanh, is the B operand of k-tile T of the next
// layer with no data movement.  The weights of all layers stay in registers.
__global__ __launch_bounds__(256) void k_mlp_infer(int64_t n, const float *__restrict__ P, const float *__restrict__ X,
                                                   float *__restrict__ Y)
{
    const int lane = threadIdx.x & 63;
    const int col = lane & 15, grp = lane >> 4;
    // weights as A operands: layer 1 (4 out tiles x 1 k tile), 2 and 3 (4 x 4), 4 (1 x 4)
    bf16x4 a1[4], a2[4][4], a3[4][4], a4[4];
    float bias1[4][4], bias2[4][4], bias3[4][4];
#pragma unroll
    for (int T = 0; T < 4; ++T) {
        const int out = 16 * T + col;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int in1 = 4 * grp + r;
            a1[T][r] = to_bf16(in1 < kMlpIn ? P[kOffW1 + in1 * kMlpW + out] : 0.0f);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int in = 16 * t + 4 * grp + r;
                a2[T][t][r] = to_bf16(P[kOffW2 + in * kMlpW + out]);
                a3[T][t][r] = to_bf16(P[kOffW3 + in * kMlpW + out]);
            }
            bias1[T][r] = P[kOffB1 + 16 * T + 4 * grp + r];
            bias2[T][r] = P[kOffB2 + 16 * T + 4 * grp + r];
            bias3[T][r] = P[kOffB3 + 16 * T + 4 * grp + r];
        }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) a4[t][r] = to_bf16(col == 0 ? P[kOffW4 + 16 * t + 4 * grp + r] : 0.0f);
    const float bias4 = P[kOffB4];

    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwave = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (int64_t g0 = wave * 16; g0 < n; g0 += nwave * 16) {
        const int64_t s = g0 + col;
        bf16x4 h[4];
        // layer 1: input features 4 grp + r of sample s
        bf16x4 x;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = 4 * grp + r;
            x[r] = to_bf16(s < n && k < kMlpIn ? X[s * kMlpInPad + k] : 0.0f);
        }
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
            d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1[T], x, d, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) h[T][r] = to_bf16(tanhf(d[r] + bias1[T][r]));
        }
        // layers 2 and 3
        bf16x4 h2[4];
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < 4; ++t) d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a2[T][t], h[t], d, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) h2[T][r] = to_bf16(tanhf(d[r] + bias2[T][r]));
        }
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < 4; ++t) d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a3[T][t], h2[t], d, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) h[T][r] = to_bf16(tanhf(d[r] + bias3[T][r]));
        }
        // layer 4: output row 0 of the single out tile sits in lanes 0..15, item 0
        f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < 4; ++t) d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a4[t], h[t], d, 0, 0, 0);
        if (grp == 0 && s < n) Y[s] = d[0] + bias4;
    }
}

// ------------------------------------------------------------------------
// the field form with the surrogate (2D)
// ------------------------------------------------------------------------
// One enumerated (grid point, bond) pair: the quadratic form of its bond
// integral (A, B; C comes with the bond entry) and the bond entry's index.
struct PairRec {
    double A, B;
    int entry;  // particle * cap + slot
    int pad;
};

// Walk the particles inside the ball of grid point t (cells around it, in
// cell order) and call visit(p, a0, a1, A) for each.
template <typename F>
__device__ __forceinline__ void for_ball(const Geom &g, const int *__restrict__ st, const double *__restrict__ sp,
                                         double x0, double x1, F &&visit)
{
    const int cx = cell_coord(g, 0, x0), cy = cell_coord(g, 1, x1);
    int rows[kMaxRows];
    const int nrows = neighbour_rows(g, cy, 0, rows);
    for (int r = 0; r < nrows; ++r) {
        int rb[2], re[2];
        const int nr = row_ranges(g, st, rows[r], cx, rb, re);
        for (int s = 0; s < nr; ++s)
            for (int p = rb[s]; p < re[s]; ++p) {
                const double a0 = minimg(sp[(size_t)p * 2] - x0, g.L[0], g.pinvL[0]);
                const double a1 = minimg(sp[(size_t)p * 2 + 1] - x1, g.L[1], g.pinvL[1]);
                const double asq = a0 * a0 + a1 * a1;
                if (asq < g.rc2) visit(p, a0, a1, asq * g.inv_rc2);
            }
    }
}

// Pairs of each grid point of one frame into counts[gp].
// The 64-bit sum of all counts goes to *total (one atomic per wavefront), so
// the host can refuse a frame whose pairs overflow the int offsets.
__global__ __launch_bounds__(128) void k_pair_count(Geom g, int G, const double *__restrict__ grid,
                                                    const int *__restrict__ st, const double *__restrict__ sp, int cap,
                                                    const int *__restrict__ bc, int *__restrict__ counts,
                                                    unsigned long long *__restrict__ total)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    int c = 0;
    if (t < G) {
        for_ball(g, st, sp, grid[(size_t)t * 3], grid[(size_t)t * 3 + 1],
                 [&](int p, double, double, double) { c += min(bc[p], cap); });
        counts[t] = c;
    }
    const unsigned long long w = wave_sum((unsigned long long)c);
    if ((threadIdx.x & 63) == 0 && w) atomicAdd(total, w);
}

// Write the pairs of grid point t at its offset (exclusive scan of the
// counts): quadratic form, entry index and the network input row.
__global__ __launch_bounds__(128) void k_pair_write(Geom g, int G, const double *__restrict__ grid,
                                                    const int *__restrict__ st, const double *__restrict__ sp, int cap,
                                                    const int *__restrict__ bc, const double *__restrict__ bd,
                                                    const int *__restrict__ offs, double rcg, PairRec *__restrict__ rec,
                                                    float *__restrict__ xin)
{
    constexpr int ES = BondLayout<2, 2, false, double>::ES;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= G) return;
    const double s2 = 2.0 * g.inv_rc;
    size_t o = (size_t)offs[t];
    for_ball(g, st, sp, grid[(size_t)t * 3], grid[(size_t)t * 3 + 1], [&](int p, double a0, double a1, double A) {
        const int nb = min(bc[p], cap);
        const double s0 = a0 * g.inv_rc, s1 = a1 * g.inv_rc;
        const double ta0 = a0 * s2, ta1 = a1 * s2;
        for (int j = 0; j < nb; ++j) {
            const double *e = bd + ((size_t)p * cap + j) * ES;
            PairRec r;
            r.A = A;
            r.B = ta0 * e[0] + ta1 * e[1];
            r.entry = p * cap + j;
            r.pad = 0;
            rec[o] = r;
            float *x = xin + o * kMlpInPad;
            x[0] = (float)s0;
            x[1] = (float)s1;
            x[2] = (float)(s0 + e[0]);
            x[3] = (float)(s1 + e[1]);
            x[4] = (float)rcg;
            x[5] = x[6] = x[7] = 0.0f;
            ++o;
        }
    });
}

// Final bond integral of each pair: the network's value where the bound of
// the pair's class (0: both ends inside the ball, so the integrand is a
// polynomial along the whole segment; 1: the segment leaves the ball) is
// within tol, the 5-node quadrature otherwise.  With tol < 0 every pair takes
// the quadrature (training targets).  Counts network pairs per workgroup.
__global__ __launch_bounds__(256) void k_pair_finalize(int64_t np, const PairRec *__restrict__ rec,
                                                       const double *__restrict__ bonds, GLRule R,
                                                       const float *__restrict__ ymlp, double bound_in,
                                                       double bound_out, double tol, double *__restrict__ w,
                                                       float *__restrict__ wf, unsigned long long *__restrict__ nmlp)
{
    constexpr int ES = BondLayout<2, 2, false, double>::ES;
    __shared__ unsigned long long sh[4];
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long used = 0;
    if (k < np) {
        const PairRec r = rec[k];
        const double *e = bonds + (size_t)r.entry * ES;
        double C = e[0] * e[0];
        C = fma(e[1], e[1], C);
        const bool inside = r.A < 1.0 && r.A + r.B + C < 1.0;
        double v;
        if (tol >= 0.0 && (inside ? bound_in : bound_out) <= tol) {
            v = (double)ymlp[k];
            used = 1;
        } else {
            v = bond_quad<0, 5, double>(R, nullptr, 5, r.A, r.B, C);
        }
        w[k] = v;
        if (wf) wf[k] = (float)v;
    }
    used = wave_sum(used);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = used;
    __syncthreads();
    if (threadIdx.x == 0 && nmlp) {
        const unsigned long long tot = sh[0] + sh[1] + sh[2] + sh[3];
        if (tot) atomicAdd(nmlp, tot);
    }
}

// Virial field of grid point t: sum over its pairs, in order, of c' w b' (x) b'.
__global__ __launch_bounds__(128) void k_pair_reduce(int G, const int *__restrict__ counts,
                                                     const int *__restrict__ offs, const PairRec *__restrict__ rec,
                                                     const double *__restrict__ bonds, const double *__restrict__ w,
                                                     double *__restrict__ out)
{
    constexpr int ES = BondLayout<2, 2, false, double>::ES;
    constexpr int OC = BondLayout<2, 2, false, double>::OC;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= G) return;
    const int c = counts[t];
    const size_t o = (size_t)offs[t];
    double v0 = 0.0, v1 = 0.0, v2 = 0.0;
    for (int k = 0; k < c; ++k) {
        const double *e = bonds + (size_t)rec[o + k].entry * ES;
        const double cw = w[o + k] * e[OC];
        const double cb0 = cw * e[0], cb1 = cw * e[1];
        v0 = fma(cb0, e[0], v0);
        v1 = fma(cb1, e[1], v1);
        v2 = fma(cb0, e[1], v2);
    }
    double *d = out + (size_t)t * 4;
    d[0] = v0;
    d[1] = v2;
    d[2] = v2;
    d[3] = v1;
}

}  // namespace pgt
