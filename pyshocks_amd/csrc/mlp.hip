// Learned WENO weights: standalone inference, the training loss and its
// gradient, the Adam update, and the learned reconstruction of a whole array.
// The perceptron and its matrix-core layout are described in mlp_device.hpp.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <string>

#include "../../include/pyshocks_amd.h"
#include "mlp_device.hpp"
#include "psa_internal.hpp"
#include "stage_device.hpp"
#include "weno5_device.hpp"

namespace psa {
namespace {

static_assert(MLP_NPARAM == PSA_MLP_NPARAM, "parameter count");

// ---------------------------------------------------------------------------
// inference on given inputs

__global__ __launch_bounds__(256) void k_mlp_weights(
    const float *__restrict__ P, const float *__restrict__ feat, long long n,
    float *__restrict__ omega, float *__restrict__ logits) {
  MlpWave W;
  mlp_load(W, P);
  const int lane = threadIdx.x & 63;
  const long long waves = static_cast<long long>(gridDim.x) * (blockDim.x >> 6);
  const long long wave = static_cast<long long>(blockIdx.x) * (blockDim.x >> 6) +
                         (threadIdx.x >> 6);
  // wave-uniform trip count: every lane of a wave runs the collective
  for (long long base = wave * 64; base < n; base += waves * 64) {
    const long long s = base + lane;
    float x[MLP_IN] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (s < n) {
#pragma unroll
      for (int k = 0; k < MLP_IN; ++k) x[k] = feat[s * MLP_IN + k];
    }
    float z[MLP_OUT], w[MLP_OUT];
    mlp_logits(W, x, z);
    mlp_softmax(z, w);
    if (s < n) {
#pragma unroll
      for (int k = 0; k < MLP_OUT; ++k) {
        omega[s * MLP_OUT + k] = w[k];
        if (logits != nullptr) logits[s * MLP_OUT + k] = z[k];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// training loss and gradient
//
// Sample record (PSA_MLP_RECORD floats): inputs x[5], normalised candidate
// errors e[3] (candidate minus exact face value, over the stencil scale),
// WENO-JS weights wjs[3], sample weight c. Loss of a sample:
//   r = sum_k omega_k e_k,  L = c (r^2 / (mean_k e_k^2 + delta)
//                               + lambda sum_k (omega_k - wjs_k)^2)
// The batch loss is the sum over samples divided by n.

constexpr int GRAD_BLOCK = 256;
constexpr int GRAD_WAVES = GRAD_BLOCK / 64;
constexpr int GRAD_CHAINS = 2;                              // of 16 samples, per wave
constexpr int GRAD_SPW = 16 * GRAD_CHAINS;                  // samples per wave
constexpr int GRAD_SAMPLES = GRAD_WAVES * GRAD_SPW;         // per workgroup and pass
constexpr int GRAD_PART = MLP_NPARAM + 1;                   // gradient entries + loss
constexpr int GRAD_MAX_BLOCKS = 1024;
constexpr int HS = MLP_HID + 1;  // padded LDS rows

typedef float f32x16_t __attribute__((ext_vector_type(16)));

// One wave's samples in FP32, a row per sample: the operands of the
// parameter-gradient products, which want a unit per lane where the passes
// over the layers leave a sample per lane.
struct GradWave {
  float h1[GRAD_SPW][HS];
  float h2[GRAD_SPW][HS];
  float dh1[GRAD_SPW][HS];
  float dh2[GRAD_SPW][HS];
  float x[GRAD_SPW][MLP_IN];
  float dz[GRAD_SPW][MLP_OUT];
};

union GradSmem {
  GradWave w[GRAD_WAVES];
  float part[GRAD_WAVES][GRAD_PART];  // the waves' sums, after the last pass
};

__device__ __forceinline__ float bf16_value(float v) {
  return static_cast<float>(static_cast<__bf16>(v));
}

// Hidden unit of k-slot j as the FP32 value of the packed BF16 activations.
__device__ __forceinline__ float slot_value(bf16x8_t h, int j) {
  return static_cast<float>(h[j]);
}

// Latency-bound at the training batch (32768 records: one workgroup per CU,
// one wave per SIMD), so the work of a wave is kept short: 32 samples as two
// independent 16-sample chains, and the parameter gradients -- sums of
// products over the samples -- on the FP32 matrix cores (exact FP32 products
// and sums: dW2 = dh2^T h1 by 16 of 32x32x2, [dW1, db1] = dh1^T [x, 1] and
// dW3 = dz^T h2 by 16x16x4) instead of a loop over the samples with one
// entry per lane. A call on 32768 records, with the reduction below: 93.6 us
// before, 11.3 us now (host launches included).
__global__ __launch_bounds__(GRAD_BLOCK) void k_mlp_grad(
    const float *__restrict__ P, const float *__restrict__ rec, long long n,
    float lambda_js, float delta, float *__restrict__ part) {
  __shared__ GradSmem sm;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int q = lane >> 4;
  const int col = lane & 15;
  GradWave &g = sm.w[wave];

  MlpWave W;
  mlp_load(W, P);
  // transposed operands of the backward products
  bf16x8_t w3t[2], w2t[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int row = 16 * b + col;  // unit of the layer below
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float a3 = (q == 0 && j < MLP_OUT) ? P[MLP_W3 + j * MLP_HID + row] : 0.0f;
      w3t[b][j] = static_cast<__bf16>(a3);
      w2t[b][j] = static_cast<__bf16>(P[MLP_W2 + mlp_slot_unit(q, j) * MLP_HID + row]);
    }
  }

  // the wave's sums: dW2 (32x32 tile), [dW1, db1] (rows 16 b + .., columns
  // 0..4 and 5), dW3 (rows 0..2, columns 16 b + ..), db2 (unit lane % 32,
  // samples of parity lane / 32), db3 and the loss (this lane's samples)
  const f32x4_t zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x16_t gW2 = {};
  f32x4_t gW1[2] = {zero4, zero4}, gW3[2] = {zero4, zero4};
  float gb2 = 0.0f, gb3[MLP_OUT] = {0.0f, 0.0f, 0.0f}, lsum = 0.0f;

  const mlp_u32x4_t none = {0u, 0u, 0u, 0u};
  for (long long base = static_cast<long long>(blockIdx.x) * GRAD_SAMPLES; base < n;
       base += static_cast<long long>(gridDim.x) * GRAD_SAMPLES) {
    const int ls = lane & (GRAD_SPW - 1);  // this lane's sample (lane < 32)
    const long long s = base + wave * GRAD_SPW + ls;
    const bool own = lane < GRAD_SPW;
    float x[MLP_IN] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    float e[3] = {0.0f, 0.0f, 0.0f}, wjs[3] = {0.0f, 0.0f, 0.0f}, c = 0.0f;
    if (own && s < n) {
      const float *r = rec + s * PSA_MLP_RECORD;
#pragma unroll
      for (int k = 0; k < MLP_IN; ++k) x[k] = r[k];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        e[k] = r[5 + k];
        wjs[k] = r[8 + k];
      }
      c = r[11];
    }
    if (own) {
#pragma unroll
      for (int k = 0; k < MLP_IN; ++k) g.x[ls][k] = bf16_value(x[k]);
    }

    // ---- forward: chain ch holds the samples of the lanes 16 ch ..
    // 16 ch + 15, whose inputs sit in k-slot group ch (see mlp_logits)
    const mlp_u32x4_t mine = mlp_pack_inputs(x);
    bf16x8_t h1[GRAD_CHAINS], h2[GRAD_CHAINS];
    float z[MLP_OUT] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ch = 0; ch < GRAD_CHAINS; ++ch) {
      const int row = 16 * ch + col;
      const bf16x8_t B = __builtin_bit_cast(bf16x8_t, q == ch ? mine : none);
      f32x4_t a0 = mlp_mfma(W.w1[0], B, W.b1[0]);
      f32x4_t a1 = mlp_mfma(W.w1[1], B, W.b1[1]);
      h1[ch] = mlp_relu_pack(a0, a1);
      a0 = mlp_mfma(W.w2[0], h1[ch], W.b2[0]);
      a1 = mlp_mfma(W.w2[1], h1[ch], W.b2[1]);
      h2[ch] = mlp_relu_pack(a0, a1);
      const f32x4_t o = mlp_mfma(W.w3, h2[ch], W.b3);
      if (q == ch) {
        z[0] = o[0];
        z[1] = o[1];
        z[2] = o[2];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        g.h1[row][mlp_slot_unit(q, j)] = slot_value(h1[ch], j);
        g.h2[row][mlp_slot_unit(q, j)] = slot_value(h2[ch], j);
      }
    }

    // ---- loss and d loss / d logits of this lane's sample (zero weight in
    // the lanes without one)
    float w[MLP_OUT];
    mlp_softmax(z, w);
    const float r = (w[0] * e[0] + w[1] * e[1]) + w[2] * e[2];
    const float den = ((e[0] * e[0] + e[1] * e[1]) + e[2] * e[2]) * (1.0f / 3.0f) + delta;
    const float inv_den = den > 0.0f ? 1.0f / den : 0.0f;
    const float dj0 = w[0] - wjs[0], dj1 = w[1] - wjs[1], dj2 = w[2] - wjs[2];
    lsum += c * (r * r * inv_den + lambda_js * ((dj0 * dj0 + dj1 * dj1) + dj2 * dj2));
    const float gr = 2.0f * c * r * inv_den;
    const float gj = 2.0f * c * lambda_js;
    const float g0 = gr * e[0] + gj * dj0;
    const float g1 = gr * e[1] + gj * dj1;
    const float g2 = gr * e[2] + gj * dj2;
    const float gw = (w[0] * g0 + w[1] * g1) + w[2] * g2;
    const float dz[MLP_OUT] = {w[0] * (g0 - gw), w[1] * (g1 - gw), w[2] * (g2 - gw)};
#pragma unroll
    for (int k = 0; k < MLP_OUT; ++k) {
      gb3[k] += dz[k];
      if (own) g.dz[ls][k] = dz[k];
    }

    // ---- backward through the hidden layers; a lane's units are the ones
    // of its packed activations, which give the ReLU masks
    const unsigned int dz01 = mlp_pack(dz[0], dz[1]), dz2 = mlp_pack(dz[2], 0.0f);
#pragma unroll
    for (int ch = 0; ch < GRAD_CHAINS; ++ch) {
      const int row = 16 * ch + col;
      // (w3t is zero outside k-slot group 0, where the column's sample goes)
      const mlp_u32x4_t zb = {__shfl(dz01, row, 64), __shfl(dz2, row, 64), 0u, 0u};
      f32x4_t d0 = mlp_mfma(w3t[0], __builtin_bit_cast(bf16x8_t, zb), zero4);
      f32x4_t d1 = mlp_mfma(w3t[1], __builtin_bit_cast(bf16x8_t, zb), zero4);
      bf16x8_t B;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        d0[v] = slot_value(h2[ch], v) > 0.0f ? d0[v] : 0.0f;
        d1[v] = slot_value(h2[ch], 4 + v) > 0.0f ? d1[v] : 0.0f;
        g.dh2[row][4 * q + v] = d0[v];
        g.dh2[row][16 + 4 * q + v] = d1[v];
        B[v] = static_cast<__bf16>(d0[v]);
        B[4 + v] = static_cast<__bf16>(d1[v]);
      }
      d0 = mlp_mfma(w2t[0], B, zero4);
      d1 = mlp_mfma(w2t[1], B, zero4);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        g.dh1[row][4 * q + v] = slot_value(h1[ch], v) > 0.0f ? d0[v] : 0.0f;
        g.dh1[row][16 + 4 * q + v] = slot_value(h1[ch], 4 + v) > 0.0f ? d1[v] : 0.0f;
      }
    }

    // ---- parameter gradients: sums over the wave's samples (its own LDS
    // rows, so the wave's own order is enough)
    wave_lds_handover();
    const int u32 = lane & 31, k2 = lane >> 5;
#pragma unroll
    for (int t = 0; t < GRAD_SPW; t += 2) {
      const float a = g.dh2[t + k2][u32];
      gb2 += a;
      gW2 = __builtin_amdgcn_mfma_f32_32x32x2f32(a, g.h1[t + k2][u32], gW2, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < GRAD_SPW; t += 4) {
      const int row = t + q;
      const float bx = col < MLP_IN ? g.x[row][col < MLP_IN ? col : 0]
                                    : (col == MLP_IN ? 1.0f : 0.0f);
      const float az = col < MLP_OUT ? g.dz[row][col < MLP_OUT ? col : 0] : 0.0f;
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        gW1[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.dh1[row][16 * b + col], bx, gW1[b],
                                                      0, 0, 0);
        gW3[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(az, g.h2[row][16 * b + col], gW3[b], 0,
                                                      0, 0);
      }
    }
    wave_lds_handover();  // (the next pass writes the rows again)
  }

  // ---- the waves' sums, then their sum in wave order
  __syncthreads();
  float *pw = sm.part[wave];
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int row = 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
    pw[MLP_W2 + row * MLP_HID + (lane & 31)] = gW2[v];
  }
#pragma unroll
  for (int b = 0; b < 2; ++b) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = 16 * b + 4 * q + v;
      if (col < MLP_IN) pw[MLP_W1 + row * MLP_IN + col] = gW1[b][v];
      if (col == MLP_IN) pw[MLP_B1 + row] = gW1[b][v];
      if (q == 0 && v < MLP_OUT) pw[MLP_W3 + v * MLP_HID + 16 * b + col] = gW3[b][v];
    }
  }
  gb2 += __shfl_xor(gb2, 32, 64);
  if (lane < MLP_HID) pw[MLP_B2 + lane] = gb2;
  for (int off = 32; off > 0; off >>= 1) {
    lsum += __shfl_xor(lsum, off, 64);
#pragma unroll
    for (int k = 0; k < MLP_OUT; ++k) gb3[k] += __shfl_xor(gb3[k], off, 64);
  }
  if (lane == 0) {
    for (int k = 0; k < MLP_OUT; ++k) pw[MLP_B3 + k] = gb3[k];
    pw[MLP_NPARAM] = lsum;
  }
  __syncthreads();
  float *out = part + static_cast<long long>(blockIdx.x) * GRAD_PART;
  for (int k = tid; k < GRAD_PART; k += GRAD_BLOCK) {
    float v = sm.part[0][k];
#pragma unroll
    for (int u = 1; u < GRAD_WAVES; ++u) v += sm.part[u][k];
    out[k] = v;
  }
}

// Sum of the block partials divided by n, in FP64: a workgroup takes 32
// entries, thread (r, e) the partials r, r + 32, .. of entry e, and the 32
// row sums are added in a fixed tree. One thread per entry over all the
// partials was a serial chain of loads: 61.8 us of those 93.6 for 256 partials.
constexpr int REDUCE_E = 32;
constexpr int REDUCE_R = 32;

__global__ __launch_bounds__(REDUCE_E *REDUCE_R) void k_mlp_grad_reduce(
    const float *__restrict__ part, int nblocks, double inv_n, float *__restrict__ grad) {
  __shared__ double s[REDUCE_R][REDUCE_E + 1];
  const int el = threadIdx.x % REDUCE_E;
  const int r = threadIdx.x / REDUCE_E;
  const int e = blockIdx.x * REDUCE_E + el;
  double acc = 0.0;
  if (e < GRAD_PART) {
#pragma unroll 4
    for (int b = r; b < nblocks; b += REDUCE_R)
      acc += part[static_cast<long long>(b) * GRAD_PART + e];
  }
  s[r][el] = acc;
  __syncthreads();
  for (int w = REDUCE_R / 2; w > 0; w >>= 1) {
    if (r < w) s[r][el] += s[r + w][el];
    __syncthreads();
  }
  if (r == 0 && e < GRAD_PART) grad[e] = static_cast<float>(s[0][el] * inv_n);
}

__global__ void k_mlp_adam(float *__restrict__ p, const float *__restrict__ g,
                           float *__restrict__ m, float *__restrict__ v, float lr,
                           float beta1, float beta2, float eps, float c1, float c2) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= MLP_NPARAM) return;
  const float ge = g[e];
  const float me = beta1 * m[e] + (1.0f - beta1) * ge;
  const float ve = beta2 * v[e] + (1.0f - beta2) * ge * ge;
  m[e] = me;
  v[e] = ve;
  p[e] -= lr * (me * c1) / (sqrtf(ve * c2) + eps);
}

// ---------------------------------------------------------------------------
// learned reconstruction of an array (the learned counterpart of
// reconstruction.py:358-377, same zero padding outside [0, m))

template <typename T>
__global__ __launch_bounds__(256) void k_learned_reconstruct(
    const float *__restrict__ P, T tau, T sigma, T eps, const T *__restrict__ u,
    T *__restrict__ ul, T *__restrict__ ur, int64_t m) {
  MlpWave W;
  mlp_load(W, P);
  const int lane = threadIdx.x & 63;
  const int64_t waves = static_cast<int64_t>(gridDim.x) * (blockDim.x >> 6);
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) +
                       (threadIdx.x >> 6);
  for (int64_t base = wave * 64; base < m; base += waves * 64) {
    const int64_t i = base + lane;
    const T um2 = load_raw(u, i - 2, m), um1 = load_raw(u, i - 1, m),
            u0 = load_raw(u, i, m), up1 = load_raw(u, i + 1, m),
            up2 = load_raw(u, i + 2, m);
    T l, r;
    learned_cell(W, um2, um1, u0, up1, up2, eps, tau, sigma, l, r);
    if (i < m) {
      ul[i] = l;
      ur[i] = r;
    }
  }
}

unsigned int grid_for(long long items, int per_block, unsigned int cap) {
  long long b = (items + per_block - 1) / per_block;
  if (b < 1) b = 1;
  if (b > cap) b = cap;
  return static_cast<unsigned int>(b);
}

}  // namespace
}  // namespace psa

using namespace psa;

extern "C" int psa_mlp_weights(const float *params, const float *features,
                               long long n, float *omega, float *logits,
                               void *stream) {
  if (n < 0) return set_error(PSA_ERR_INVALID_ARGUMENT, "negative sample count");
  if (n == 0) return PSA_OK;
  if (params == nullptr || features == nullptr || omega == nullptr)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "null pointer");
  hipLaunchKernelGGL(k_mlp_weights, dim3(grid_for(n, 256, 4096)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), params, features, n, omega,
                     logits);
  return check_launch("mlp weights");
}

extern "C" int psa_mlp_grad_workspace_bytes(long long n, size_t *bytes) {
  if (n < 0 || bytes == nullptr)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "bad arguments");
  const unsigned int nb = grid_for(n, GRAD_SAMPLES, GRAD_MAX_BLOCKS);
  *bytes = static_cast<size_t>(nb) * GRAD_PART * sizeof(float);
  return PSA_OK;
}

extern "C" int psa_mlp_grad(const float *params, const float *samples, long long n,
                            double lambda_js, double delta, float *grad, void *work,
                            size_t work_bytes, void *stream) {
  if (n <= 0) return set_error(PSA_ERR_INVALID_ARGUMENT, "no samples");
  if (params == nullptr || samples == nullptr || grad == nullptr || work == nullptr)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "null pointer");
  if (!(lambda_js >= 0.0) || !(delta >= 0.0))
    return set_error(PSA_ERR_INVALID_ARGUMENT, "lambda and delta must be >= 0");
  const unsigned int nb = grid_for(n, GRAD_SAMPLES, GRAD_MAX_BLOCKS);
  if (work_bytes < static_cast<size_t>(nb) * GRAD_PART * sizeof(float))
    return set_error(PSA_ERR_WORKSPACE, "gradient workspace too small");
  auto s = static_cast<hipStream_t>(stream);
  float *part = static_cast<float *>(work);
  hipLaunchKernelGGL(k_mlp_grad, dim3(nb), dim3(GRAD_BLOCK), 0, s, params, samples, n,
                     static_cast<float>(lambda_js), static_cast<float>(delta), part);
  int st = check_launch("mlp gradient");
  if (st != PSA_OK) return st;
  hipLaunchKernelGGL(k_mlp_grad_reduce, dim3((GRAD_PART + REDUCE_E - 1) / REDUCE_E),
                     dim3(REDUCE_E * REDUCE_R), 0, s, part, static_cast<int>(nb), 1.0 / static_cast<double>(n), grad);
  return check_launch("mlp gradient reduce");
}

extern "C" int psa_mlp_adam(float *params, const float *grad, float *m, float *v,
                            long long step, double lr, double beta1, double beta2,
                            double eps, void *stream) {
  if (params == nullptr || grad == nullptr || m == nullptr || v == nullptr)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "null pointer");
  if (step < 1 || !(lr > 0.0) || !(beta1 >= 0.0 && beta1 < 1.0) ||
      !(beta2 >= 0.0 && beta2 < 1.0) || !(eps > 0.0))
    return set_error(PSA_ERR_INVALID_ARGUMENT, "bad Adam parameters");
  const double c1 = 1.0 / (1.0 - std::pow(beta1, static_cast<double>(step)));
  const double c2 = 1.0 / (1.0 - std::pow(beta2, static_cast<double>(step)));
  hipLaunchKernelGGL(k_mlp_adam, dim3((MLP_NPARAM + 255) / 256), dim3(256), 0,
                     static_cast<hipStream_t>(stream), params, grad, m, v,
                     static_cast<float>(lr), static_cast<float>(beta1),
                     static_cast<float>(beta2), static_cast<float>(eps),
                     static_cast<float>(c1), static_cast<float>(c2));
  return check_launch("mlp adam");
}

extern "C" int psa_learned_reconstruct(int dtype, const float *params, double tau,
                                       double sigma, const void *u, void *ul, void *ur,
                                       int64_t m, double eps, void *stream) {
  if (m < 0) return set_error(PSA_ERR_INVALID_ARGUMENT, "negative size");
  if (m == 0) return PSA_OK;
  if (params == nullptr || u == nullptr || ul == nullptr || ur == nullptr)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "null pointer");
  if (!(tau >= 0.0) || !(sigma >= 0.0) || !(eps >= 0.0))
    return set_error(PSA_ERR_INVALID_ARGUMENT, "tau, sigma and eps must be >= 0");
  auto s = static_cast<hipStream_t>(stream);
  const unsigned int nb = grid_for(m, 256, 4096);
  if (dtype == PSA_FLOAT64) {
    hipLaunchKernelGGL(k_learned_reconstruct<double>, dim3(nb), dim3(256), 0, s, params,
                       tau, sigma, eps, static_cast<const double *>(u),
                       static_cast<double *>(ul), static_cast<double *>(ur), m);
  } else if (dtype == PSA_FLOAT32) {
    hipLaunchKernelGGL(k_learned_reconstruct<float>, dim3(nb), dim3(256), 0, s, params,
                       static_cast<float>(tau), static_cast<float>(sigma),
                       static_cast<float>(eps),
                       static_cast<const float *>(u), static_cast<float *>(ul),
                       static_cast<float *>(ur), m);
  } else {
    return set_error(PSA_ERR_NOT_IMPLEMENTED, "unsupported dtype");
  }
  return check_launch("learned reconstruct");
}
