// Discrete adjoint (vector-Jacobian products) of the fused SSP-RK3 step.
//
// The reference differentiates one step with a dense forward-mode Jacobian
// (timestepping.py:155-215, jax.jacfwd of advance). Here the transposed
// Jacobian is applied matrix-free, one reverse kernel per Runge-Kutta stage:
//
//   forward  k1 = x + dt L(x)
//            k2 = 3/4 x + 1/4 (k1 + dt L(k1))
//            x+ = 1/3 x + 2/3 (k2 + dt L(k2))
//   reverse  lk2 = 2/3 (l + dt JL(k2)^T l)
//            lk1 = 1/4 (lk2 + dt JL(k1)^T lk2)
//            lx  = 1/3 l + 3/4 lk2 + lk1 + dt JL(x)^T lk1
//
// JL^T mu is formed per cell from the closed-form gradient of the two WENO-JS5
// reconstructions of the cell and the partial derivatives of the face flux.
// Derivative conventions at the non-smooth points follow jax: jnp.maximum
// splits a tie 0.5 / 0.5, d|u|/du = sign(u) with sign(0) = 0, and the upwind
// selection (jnp.where) passes the derivative of the selected branch only.
// dt is a constant (adjoint_step recovers it as t_{m+1} - t_m).
//
// The state and the cotangents are periodic: every index is mapped to its
// interior image, which also covers the 5-cell halo the transpose needs.
//
// Learned weights (LEARNED kernels): each cell takes its forward regime (from
// the same fused indicator arithmetic as the forward kernels); shock cells
// differentiate WENO-JS, smooth cells the ideal weights, learned cells the
// network. The network is differentiated as the smooth function it rounds:
// BF16 parameters (as the forward's operands), inputs and activations
// unrounded, in the state dtype -- the adjoint of that surrogate along the
// forward's trajectory.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>

#include "../../include/pyshocks_amd.h"
#include "mlp_device.hpp"
#include "psa_internal.hpp"
#include "stage_device.hpp"
#include "weno5_device.hpp"

namespace psa {
namespace {

constexpr int kVjpBlock = 256;          // threads and computing cells per workgroup
constexpr int kVjpWaves = kVjpBlock / 64;
constexpr int kVjpOut = kVjpBlock - 6;  // output cells per workgroup
constexpr int kVjpMostSteps = 12;       // reverse steps of a launch (40 output cells)

// 1 / x for a positive normal FP64 x: the hardware reciprocal y (relative
// error e below 1e-7) with e + e^2 added, which leaves e^3.
__device__ __forceinline__ double rcp_refined(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);
  return fma(y, fma(e, e, e), y);
}

// Both reconstructions of a cell and what their gradients take. The forward
// kernels' difference form: D_k the first differences of the stencil, s_k the
// second ones, t = (2 D1 + s0, D1 + D2, s2 - 2 D2), e_k = 4 (eps + beta_k) =
// 4 eps + 13/3 s_k^2 + t_k^2, T0 = s1 - s0, T1 = s2 - s1;
//   hR_0, hR_1, hR_2 = u + (2 t0 - D1, t1 + D2, D2 - t2) / 6,
//   hL_0, hL_1, hL_2 = u - (t0 + D1, t1 + D1, -2 t2 - D2) / 6,
// the weights indexed by their indicator: wR_k ~ (1, 6, 3) / e_k^2, wL_k ~
// (3, 6, 1) / e_k^2, normalised. With
//   dur/de_k = -2 zR_k,  zR_k = wR_k (hR_k - ur) / e_k   (left alike)
// the two sides share everything up to the weights, and their contributions
// meet in one set of derivatives of e_k (weno_cell_scatter).
template <typename T>
struct CellStates {
  T s[3], t[3];
  T qR[3], qL[3];  // 6 w_k (h_k - value) of the right and left state
  T ie[3];         // 1 / e_k
  T wR0, wR2, wL0, wL2;
};

// The weights of both sides and 1 / e_k. FP64: one refined reciprocal of
// e0 e1 e2 and one of the product of the two weight sums where both are
// positive normal numbers, else the divisions; FP32: the divisions.
template <typename T>
__device__ __forceinline__ void weno_cell_weights(T e0, T e1, T e2, T ie[3], T wR[3],
                                                  T wL[3]) {
  bool fast = false;
  if constexpr (std::is_same<T, double>::value) {
    const double e01 = e0 * e1, e12 = e1 * e2, e02 = e0 * e2;
    const double den = e01 * e2;
    const double inv = rcp_refined(den);
    ie[0] = e12 * inv;
    ie[1] = e02 * inv;
    ie[2] = e01 * inv;
    const double x0 = ie[0] * ie[0], x1 = 6.0 * (ie[1] * ie[1]), x2 = ie[2] * ie[2];
    const double aR = fma(3.0, x2, x0 + x1), aL = fma(3.0, x0, x2 + x1);
    const double aa = aR * aL;
    const double ia = rcp_refined(aa);
    const double iR = aL * ia, iL = aR * ia;
    wR[0] = x0 * iR;
    wR[1] = x1 * iR;
    wR[2] = 3.0 * (x2 * iR);
    wL[0] = 3.0 * (x0 * iL);
    wL[1] = x1 * iL;
    wL[2] = x2 * iL;
    fast = __builtin_amdgcn_class(den, 0x100) && __builtin_amdgcn_class(aa, 0x100);
  }
  if (__builtin_expect(!fast, std::is_same<T, float>::value)) {
    using C = Weno5Coeffs<T>;
    // (of eps + beta_k, a quarter: the squares' range)
    const T f0 = T(0.25) * e0, f1 = T(0.25) * e1, f2 = T(0.25) * e2;
    const T q0 = f0 * f0, q1 = f1 * f1, q2 = f2 * f2;
    const T a0 = C::d0 / q0, a1 = C::d1 / q1, a2 = C::d2 / q2;
    const T l0 = C::d2 / q0, l2 = C::d0 / q2;
    const T aR = (a0 + a1) + a2, aL = (l2 + a1) + l0;
    wR[0] = a0 / aR;
    wR[1] = a1 / aR;
    wR[2] = a2 / aR;
    wL[0] = l0 / aL;
    wL[1] = a1 / aL;
    wL[2] = l2 / aL;
    ie[0] = T(1) / e0;
    ie[1] = T(1) / e1;
    ie[2] = T(1) / e2;
  }
}

// The differences of the stencil (into c.s, c.t) and the indicators e_k.
template <typename T>
__device__ __forceinline__ void weno_cell_indicators(const T v[5], T eps4, T &D1, T &D2,
                                                     CellStates<T> &c, T e[3]) {
  using C = Weno5Coeffs<T>;
  const T D0 = v[1] - v[0];
  D1 = v[2] - v[1];
  D2 = v[3] - v[2];
  const T D3 = v[4] - v[3];
  c.s[0] = D1 - D0;
  c.s[1] = D2 - D1;
  c.s[2] = D3 - D2;
  c.t[0] = fma(T(2), D1, c.s[0]);
  c.t[1] = D2 + D1;
  c.t[2] = fma(T(-2), D2, c.s[2]);
#pragma unroll
  for (int k = 0; k < 3; ++k)
    e[k] = fma(c.t[k], c.t[k], fma(C::a0x4, c.s[k] * c.s[k], eps4));
}

// Both states from the middle candidates and the weights c.wR0 .. c.wL2 (the
// learned kernels' form, mlp_combine_ideal).
template <typename T>
__device__ __forceinline__ void weno_cell_values(T u, T D1, T D2, const CellStates<T> &c,
                                                 T &ul, T &ur) {
  const T a = (c.s[1] - c.s[0]) * T(1.0 / 6.0), b = (c.s[2] - c.s[1]) * T(1.0 / 6.0);
  const T mR = fma(c.wR0, a + a, c.wR2 * b);
  const T mL = fma(c.wL2, b + b, c.wL0 * a);
  ur = fma(c.t[1] + D2, T(1.0 / 6.0), u) - mR;
  ul = fma(c.t[1] + D1, T(-1.0 / 6.0), u) + mL;
}

// WENO-JS states of a cell from its stencil and what the gradient takes.
template <typename T>
__device__ __forceinline__ void weno_cell_states(const T v[5], T eps4, CellStates<T> &c,
                                                 T &ul, T &ur) {
  T D1, D2, e[3], wR[3], wL[3];
  weno_cell_indicators(v, eps4, D1, D2, c, e);
  weno_cell_weights(e[0], e[1], e[2], c.ie, wR, wL);
  c.wR0 = wR[0];
  c.wR2 = wR[2];
  c.wL0 = wL[0];
  c.wL2 = wL[2];
  // the states: the cell's value plus a convex sum of the candidates' distances
  // from it, so that a candidate across a jump enters with its weight only
  const T dR = fma(wR[2], D2 - c.t[2], fma(wR[1], c.t[1] + D2, wR[0] * fma(T(2), c.t[0], -D1)));
  const T dL = fma(wL[2], fma(T(-2), c.t[2], -D2), fma(wL[1], c.t[1] + D1, wL[0] * (c.t[0] + D1)));
  ur = fma(dR, T(1.0 / 6.0), v[2]);
  ul = fma(dL, T(-1.0 / 6.0), v[2]);
  // 6 (h_k - value) as sums of weighted differences of the candidates, 6 (hR_0 -
  // hR_1) = -2 T0, 6 (hR_2 - hR_1) = -T1, 6 (hL_0 - hL_1) = T0, 6 (hL_2 - hL_1) =
  // 2 T1: every term across a jump carries the weight that makes it small (the
  // difference of a candidate and the state would leave a rounding of the jump,
  // and 1 / e_k magnifies it); the middle one from their sum, which is zero
  const T T0 = c.s[1] - c.s[0], T1 = c.s[2] - c.s[1];
  const T r = fma(T(-2), T0, T1), l = fma(T(-2), T1, T0);
  c.qR[0] = wR[0] * fma(wR[2], r, -(wR[1] * (T0 + T0)));
  c.qR[2] = -(wR[2] * fma(wR[0], r, wR[1] * T1));
  c.qR[1] = -(c.qR[0] + c.qR[2]);
  c.qL[0] = wL[0] * fma(wL[2], l, wL[1] * T0);
  c.qL[2] = wL[2] * fma(wL[1], T1 + T1, -(wL[0] * l));
  c.qL[1] = -(c.qL[0] + c.qL[2]);
}

// cR dur/dv + cL dul/dv of a cell: through the weights (z_k = (cR qR_k +
// cL qL_k) / e_k, de_k = 26/3 s_k ds_k + 2 t_k dt_k; none with FIXED, weights
// that do not depend on v), through T0 and T1 at fixed weights and through the
// middle candidates, from the second to the first differences and to v.
template <typename T>
__device__ __forceinline__ void weno_cell_scatter(const CellStates<T> &c, T cR, T cL,
                                                  bool fixed, T P[5]) {
  T at[3], as[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const T z = fixed ? T(0)
                      : T(-2.0 / 3.0) * (fma(cR, c.qR[k], cL * c.qL[k]) * c.ie[k]);
    at[k] = z * c.t[k];
    as[k] = T(13.0 / 3.0) * (z * c.s[k]);
  }
  const T aT0 = fma(T(-2) * cR, c.wR0, cL * c.wL0) * T(1.0 / 6.0);
  const T aT1 = fma(T(2) * cL, c.wL2, -(cR * c.wR2)) * T(1.0 / 6.0);
  as[0] = (as[0] - aT0) + at[0];
  as[1] = as[1] + (aT0 - aT1);
  as[2] = (as[2] + aT1) + at[2];
  const T h = (cR - cL) * T(1.0 / 6.0);
  // cR/6 - cL/3 = h - cL/6, cR/3 - cL/6 = h + cR/6
  const T g1 = (as[0] - as[1]) + (fma(T(2), at[0], at[1]) + fma(T(-1.0 / 6.0), cL, h));
  const T g2 = (as[1] - as[2]) + (fma(T(-2), at[2], at[1]) + fma(T(1.0 / 6.0), cR, h));
  // v_k: D_{k-1} + ... (D0 takes -as0, D3 takes as2)
  P[0] = as[0];
  P[1] = -as[0] - g1;
  P[2] = (g1 - g2) + (cR + cL);
  P[3] = g2 - as[2];
  P[4] = as[2];
}

template <typename T>
__device__ __forceinline__ T sgn(T x) {
  return x > T(0) ? T(1) : (x < T(0) ? T(-1) : T(0));
}

template <typename T>
struct VjpArgs {
  const T *state;   // stencil input of the forward stage
  const T *mu;      // cotangent of the stage operator output
  const T *lam;     // RSTAGE 1: cotangent of the step output
  const T *lamk2;   // RSTAGE 1: cotangent of k2
  T *out;
  const T *dt_ptr;
  int64_t m;
  int64_t n;
  int g;
  T inv_dx;
  T eps;
  T vconst;
  const float *mlp;   // LEARNED: the network's parameters (PSA_MLP_NPARAM FP32)
  T eps4;             // 4 eps (the indicators carry 4 beta)
  T tau;              // LEARNED: shock threshold
  T sigma;            // LEARNED: smooth threshold
  T alpha;            // Lax-Friedrichs: the global speed max|state| (in-kernel)
};

// A weight as the forward kernels' BF16 operand (round to nearest even, on
// the bit pattern: the parameters are uniform, so this stays in scalar
// registers), as the state dtype.
template <typename T>
__device__ __forceinline__ T mlp_weight(const float *__restrict__ P, int i);

template <>
__device__ __forceinline__ float mlp_weight<float>(const float *__restrict__ P, int i) {
  unsigned int b = __float_as_uint(P[i]);
  b = (b + 0x7FFFu + ((b >> 16) & 1u)) & 0xFFFF0000u;
  return __uint_as_float(b);
}

// FP64: the BF16 value's exact FP64 bits built from its FP32 bits (sign,
// exponent rebiased by 1023 - 127, the 7 mantissa bits; BF16 values below
// the FP32 normal range are taken as zero), so that the weight stays a
// scalar operand of the multiply-adds.
template <>
__device__ __forceinline__ double mlp_weight<double>(const float *__restrict__ P, int i) {
  unsigned int b = __float_as_uint(P[i]);
  b = (b + 0x7FFFu + ((b >> 16) & 1u)) & 0xFFFF0000u;
  const unsigned int e = (b >> 23) & 0xFFu;
  const unsigned int hi =
      e == 0u ? (b & 0x80000000u)
              : ((b & 0x80000000u) | ((e + 896u) << 20) | ((b >> 3) & 0x000FFFFFu));
  return __hiloint2double(static_cast<int>(hi), 0);
}

// The network of the learned kernels in LDS, its weights as the forward
// kernels round them (mlp_weight) and b3 + ln d summed in FP32 as the
// forward's accumulator start, with room for one layer of the two sides that a
// wave evaluates at once and the list of the workgroup's learned cells.
template <typename T, bool USED>
struct VjpNet {
  int count;
  unsigned short cell[kVjpBlock];
  T w1[MLP_HID][MLP_IN], b1[MLP_HID];
  T w2[MLP_HID][MLP_HID + 1], b2[MLP_HID];
  T w3[MLP_OUT][MLP_HID], b3[MLP_OUT + 1];
  __align__(16) T h[kVjpWaves][2][MLP_HID];
};
template <typename T>
struct VjpNet<T, false> {};

// Fills the network (a barrier must follow).
template <typename T>
__device__ __forceinline__ void vjp_net_load(VjpNet<T, true> &net,
                                             const float *__restrict__ P) {
  const int tid = threadIdx.x;
  if (tid == 0) net.count = 0;
  for (int i = tid; i < MLP_HID * MLP_HID; i += kVjpBlock)
    net.w2[i / MLP_HID][i % MLP_HID] = mlp_weight<T>(P, MLP_W2 + i);
  if (tid < MLP_HID * MLP_IN) net.w1[tid / MLP_IN][tid % MLP_IN] = mlp_weight<T>(P, MLP_W1 + tid);
  if (tid < MLP_OUT * MLP_HID)
    net.w3[tid / MLP_HID][tid % MLP_HID] = mlp_weight<T>(P, MLP_W3 + tid);
  if (tid < MLP_HID) {
    net.b1[tid] = static_cast<T>(P[MLP_B1 + tid]);
    net.b2[tid] = static_cast<T>(P[MLP_B2 + tid]);
  }
  const float lnd[3] = {MLP_LN_D0, MLP_LN_D1, MLP_LN_D2};
#pragma unroll
  for (int o = 0; o < MLP_OUT; ++o)
    if (tid == o) net.b3[o] = static_cast<T>(P[MLP_B3 + o] + lnd[o]);
}

// Sum over the 32 lanes of each half of the wave, to every lane of the half:
// DPP moves within the rows of 16 lanes, a swizzle between the two rows.
template <int CTRL>
__device__ __forceinline__ float dpp_value(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_value(double v) {
  return __hiloint2double(
      __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true),
      __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float other_row(float v) {  // lane ^ 16
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401F));
}
__device__ __forceinline__ double other_row(double v) {
  return __hiloint2double(__builtin_amdgcn_ds_swizzle(__double2hiint(v), 0x401F),
                          __builtin_amdgcn_ds_swizzle(__double2loint(v), 0x401F));
}
template <typename T>
__device__ __forceinline__ T half_sum(T v) {
  v += dpp_value<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dpp_value<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_value<0x141>(v);  // row_half_mirror
  v += dpp_value<0x140>(v);  // row_mirror
  return v + other_row(v);
}

// The normalised inputs x = (v - mean) / s of the network, s = |d_km| =
// max|d|, d = v - mean; inv = 1 / s (0 where s = 0), sg = sgn(d_km).
template <typename T>
__device__ __forceinline__ void learned_inputs(const T v[5], T x[5], T &inv, T &sg, int &km) {
  const T mean = (((v[0] + v[4]) + (v[1] + v[3])) + v[2]) * T(0.2);
  T s = T(0);
  sg = T(-1);
  km = 0;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    x[k] = v[k] - mean;
    if (fabs(x[k]) > s) {
      s = fabs(x[k]);
      sg = x[k] > T(0) ? T(1) : T(-1);
      km = k;
    }
  }
  inv = s > T(0) ? T(1) / s : T(0);
#pragma unroll
  for (int k = 0; k < 5; ++k) x[k] = x[k] * inv;
}

// The network on the cell whose stencil starts at v (in LDS, the same cell in
// every lane): weights w0, w2 and, of the reconstructed value r = h1 +
// w0 (h0 - h1) + w2 (h2 - h1), w = softmax(z), the gradient xb with respect to
// the inputs, back through softmax and the three layers (ReLU masks of this
// evaluation). The lanes 0 .. 31 are the hidden units of the right side, the
// lanes 32 .. 63 those of the left side (the mirrored stencil); a layer's
// values pass through LDS, sums over units through DPP.
template <typename T>
__device__ __forceinline__ void learned_network(VjpNet<T, true> &net, const T *s_v, T &p0,
                                                T &p2, T xb[5]) {
  const int lane = threadIdx.x & 63;
  const int unit = lane & 31;
  const bool left = lane >= 32;
  T *hb = net.h[threadIdx.x >> 6][left ? 1 : 0];
  const T v[5] = {s_v[0], s_v[1], s_v[2], s_v[3], s_v[4]};
  T x[5], inv, sg;
  int km;
  learned_inputs(v, x, inv, sg, km);
  const T D0 = v[1] - v[0], D1 = v[2] - v[1], D2 = v[3] - v[2], D3 = v[4] - v[3];
  const T s0 = D1 - D0, s1 = D2 - D1, s2 = D3 - D2;
  const T t0 = s1 - s0, t1 = s2 - s1;

  // forward
  T w1[MLP_IN], w3[MLP_OUT];
#pragma unroll
  for (int k = 0; k < MLP_IN; ++k) w1[k] = net.w1[unit][k];
#pragma unroll
  for (int o = 0; o < MLP_OUT; ++o) w3[o] = net.w3[o][unit];
  T a1 = net.b1[unit];
#pragma unroll
  for (int k = 0; k < 5; ++k) a1 = fma(w1[k], left ? x[4 - k] : x[k], a1);
  hb[unit] = a1 > T(0) ? a1 : T(0);
  wave_lds_handover();
  T acc[4] = {net.b2[unit], T(0), T(0), T(0)};
#pragma unroll 8
  for (int j = 0; j < MLP_HID; ++j) acc[j & 3] = fma(net.w2[unit][j], hb[j], acc[j & 3]);
  const T a2 = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  const T h2 = a2 > T(0) ? a2 : T(0);
  T z[MLP_OUT];
#pragma unroll
  for (int o = 0; o < MLP_OUT; ++o) z[o] = half_sum(w3[o] * h2) + net.b3[o];
  const T zm = fmax(fmax(z[0], z[1]), z[2]);
  const T e0 = exp(z[0] - zm), e1 = exp(z[1] - zm), e2 = exp(z[2] - zm);
  const T es = T(1) / ((e0 + e1) + e2);
  p0 = e0 * es;
  p2 = e2 * es;
  const T p1 = e1 * es;

  // backward: dr/dw = (h0 - h1, 0, h2 - h1), through softmax
  const T c0 = left ? t1 * T(1.0 / 3.0) : t0 * T(-1.0 / 3.0);
  const T c2 = left ? t0 * T(1.0 / 6.0) : t1 * T(-1.0 / 6.0);
  const T sw = c0 * p0 + c2 * p2;
  const T hb2 =
      fma(w3[0], p0 * (c0 - sw), fma(w3[1], p1 * (T(0) - sw), w3[2] * (p2 * (c2 - sw))));
  wave_lds_handover();
  hb[unit] = a2 > T(0) ? hb2 : T(0);
  wave_lds_handover();
  T bcc[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll 8
  for (int i = 0; i < MLP_HID; ++i) bcc[i & 3] = fma(net.w2[i][unit], hb[i], bcc[i & 3]);
  T hb1 = (bcc[0] + bcc[1]) + (bcc[2] + bcc[3]);
  hb1 = a1 > T(0) ? hb1 : T(0);
#pragma unroll
  for (int k = 0; k < 5; ++k) xb[k] = half_sum(w1[k] * hb1);
  wave_lds_handover();
}

// What the network adds to the states of the learned cells of a workgroup:
// the weights of both sides (into c: wR = (w0, ., w2), wL likewise, mirrored)
// and the gradients gR, gL of the states through the weights, on the
// (unmirrored) stencil. s_u: the states, cell t's stencil at s_u[t]; res:
// kLearnedRound * 14 values of LDS scratch. Ends a barrier after its first
// reads of net.count.
//
// The learned cells sit together around jumps and critical points, ten or
// twenty of them in one or two waves of a grid. They are collected for the
// workgroup and dealt to its waves, and a wave evaluates one with a lane per
// hidden unit: with a lane per cell that walked the network alone, a stage
// waited for two serial loops over its rows and a reverse step of 16
// instances of 16384 cells took 377 us.
constexpr int kLearnedRound = 64;  // cells per round

template <typename T>
__device__ __forceinline__ void learned_cells_grad(VjpNet<T, true> &net, bool learned,
                                                   const T *s_u, const T v[5], T *res,
                                                   CellStates<T> &c, T gR[5], T gL[5]) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const unsigned long long mine = __ballot(learned);
  int slot = 0;
  if (mine != 0) {  // wave-uniform
    int base = 0;
    if (lane == 0) base = atomicAdd(&net.count, __popcll(mine));
    slot = __builtin_amdgcn_readfirstlane(base) +
           __popcll(mine & ((1ull << lane) - 1ull));
    if (learned) net.cell[slot] = static_cast<unsigned short>(tid);
  }
  __syncthreads();
  const int total = __builtin_amdgcn_readfirstlane(net.count);
  if (total == 0) return;  // workgroup-uniform
  for (int r0 = 0; r0 < total; r0 += kLearnedRound) {
    const int end = total - r0 < kLearnedRound ? total - r0 : kLearnedRound;
    for (int e = tid >> 6; e < end; e += kVjpWaves) {
      const int cell = __builtin_amdgcn_readfirstlane(net.cell[r0 + e]);
      T p0, p2, xb[5];
      learned_network(net, s_u + cell, p0, p2, xb);
      if ((lane & 31) == 0) {
        T *out = res + 14 * e + (lane >= 32 ? 7 : 0);
        out[0] = p0;
        out[1] = p2;
#pragma unroll
        for (int k = 0; k < 5; ++k) out[2 + k] = xb[k];
      }
    }
    __syncthreads();
    if (learned && slot >= r0 && slot < r0 + end) {
      const T *in = res + 14 * (slot - r0);
      c.wR0 = in[0];
      c.wR2 = in[1];
      c.wL2 = in[7];
      c.wL0 = in[8];
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        gR[k] = in[2 + k];
        gL[k] = in[13 - k];  // back on the unmirrored stencil
      }
    }
    if (r0 + kLearnedRound < total) __syncthreads();
  }

  // from the inputs to the stencil: x_k = d_k / s with d = v - mean and s =
  // |d_km|: dx_k/dv_j = (delta_kj - 1/5) / s - x_k sgn(d_km) (delta_km,j - 1/5) / s
  if (learned) {
    T x[5], inv, sg;
    int km;
    learned_inputs(v, x, inv, sg, km);
    T sr = T(0), sl = T(0), dr = T(0), dl = T(0);
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      sr += gR[k];
      sl += gL[k];
      dr += gR[k] * x[k];
      dl += gL[k] * x[k];
    }
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      const T ds = sg * ((j == km ? T(1) : T(0)) - T(0.2));
      gR[j] = inv * ((gR[j] - T(0.2) * sr) - dr * ds);
      gL[j] = inv * ((gL[j] - T(0.2) * sl) - dl * ds);
    }
  }
}

// Scratch of one reverse stage over a block of kVjpBlock computing cells.
template <typename T, bool LEARNED>
struct VjpScratch {
  T ul[kVjpBlock];
  T cL[kVjpBlock], sR[kVjpBlock];
  T P[5][kVjpBlock];
  VjpNet<T, LEARNED> net;
};

// JL(state)^T mu for the output cells Z .. Z + B - 7 of one block: s_u holds
// the state at cells Z - 5 .. Z + B - 2, s_mu the cotangent at Z - 3 ..
// Z + B - 3 (both in LDS, visible to the block). Thread t computes both
// reconstructions of cell Z - 3 + t, the face to its right, and its
// contributions to the five cells around it; it returns the gathered sum of
// output cell Z + t (valid for t < B - 6). s_u is read only before the second
// barrier (a caller may overwrite it once this returns). Ends with the scratch
// in use.
//
// VALU-bound in a batch, latency-bound for one instance. Both sides in one
// thread share the indicators and reciprocals, and their gradients are expanded
// to the stencil once, after the faces have given both cotangents; two threads
// per cell with a gradient each took 49.7 us (in one thread; 64 instances of
// 16384 cells) and 7.96 us (in two; one instance) per reverse step.
template <typename T, int FLUX, bool LEARNED = false>
__device__ __forceinline__ T vjp_block(const VjpArgs<T> &p, const T *s_u,
                                       const T *s_mu, VjpScratch<T, LEARNED> &sc) {
  constexpr int B = kVjpBlock;
  const int tid = threadIdx.x;

  // ---- both states of computing cell Z - 3 + tid
  const T v[5] = {s_u[tid], s_u[tid + 1], s_u[tid + 2], s_u[tid + 3], s_u[tid + 4]};
  CellStates<T> c;
  T ul, ur;
  int regime = 0;
  T gR[LEARNED ? 5 : 1] = {}, gL[LEARNED ? 5 : 1] = {};
  if constexpr (LEARNED) {
    // the forward kernels' regime, from their arithmetic (reconstruct_cells)
    using C = Weno5Coeffs<T>;
    T D1, D2, e[3];
    weno_cell_indicators(v, p.eps4, D1, D2, c, e);
    regime = mlp_regime(fma(c.t[0], c.t[0], C::a0x4 * (c.s[0] * c.s[0])),
                        fma(c.t[1], c.t[1], C::a0x4 * (c.s[1] * c.s[1])),
                        fma(c.t[2], c.t[2], C::a0x4 * (c.s[2] * c.s[2])), p.eps4, p.tau,
                        p.sigma);
    c.wR0 = c.wL2 = T(0.1);
    c.wR2 = c.wL0 = T(0.3);
    static_assert(5 * B >= 14 * kLearnedRound, "the scatter's scratch holds a round");
    learned_cells_grad(sc.net, regime == 2, s_u, v, &sc.P[0][0], c, gR, gL);
    weno_cell_values(v[2], D1, D2, c, ul, ur);
    if (regime == 0) weno_cell_states(v, p.eps4, c, ul, ur);
  } else {
    weno_cell_states(v, p.eps4, c, ul, ur);
  }
  sc.ul[tid] = ul;
  __syncthreads();
  if constexpr (LEARNED) {
    // (the next stage adds to it after the barriers below)
    if (tid == 0) sc.net.count = 0;
  }

  // ---- the face right of the cell: cotangent of the flux and its partial
  // derivatives (cR, sL stay here, cL and sR go to the next cell)
  T cR = T(0), sL = T(0);
  if (tid < B - 1) {
    const T urL = ur, ulR = sc.ul[tid + 1];
    const T uL = v[2], uR = v[3];
    T gF = (s_mu[tid + 1] - s_mu[tid]) * p.inv_dx;
    T dur = T(0), dul = T(0), duL = T(0), duR = T(0);
    if constexpr (FLUX == PSA_FLUX_RUSANOV) {
      // F = 0.5 (ul^2/2 + ur^2/2) - 0.5 a (ul - ur), a = max(|uR|, |uL|)
      const T aR = fabs(uR), aL = fabs(uL);
      const T a = aR > aL ? aR : aL;
      dur = T(0.5) * urL + T(0.5) * a;
      dul = T(0.5) * ulR - T(0.5) * a;
      const T dFda = T(-0.5) * (ulR - urL);
      const T wR = aR > aL ? T(1) : (aR < aL ? T(0) : T(0.5));
      duR = dFda * wR * sgn(uR);
      duL = dFda * (T(1) - wR) * sgn(uL);
    } else if constexpr (FLUX == PSA_FLUX_LAX_FRIEDRICHS) {
      // F = 0.5 (ul^2/2 + ur^2/2) - 0.5 alpha (ul - ur) with the global speed
      // alpha, whose own derivative k_lf_speed_vjp adds
      dur = T(0.5) * urL + T(0.5) * p.alpha;
      dul = T(0.5) * ulR - T(0.5) * p.alpha;
    } else if constexpr (FLUX == PSA_FLUX_ENGQUIST_OSHER) {
      // F = max(ur, 0)^2 / 2 + min(ul, 0)^2 / 2
      dur = urL > T(0) ? urL : T(0);
      dul = ulR < T(0) ? ulR : T(0);
    } else if constexpr (FLUX == PSA_FLUX_BURGERS_UPWIND) {
      const T aavg = (urL + ulR) / T(2);
      if (aavg > T(0)) {
        dur = urL;
      } else {
        dul = ulR;
      }
    } else {
      // constant velocity a: L = -a (F[1:] - F[:-1]) / dx, F = ur if a > 0
      gF *= p.vconst;
      if (p.vconst > T(0)) {
        dur = T(1);
      } else {
        dul = T(1);
      }
    }
    cR = gF * dur;
    sL = gF * duL;
    sc.cL[tid + 1] = gF * dul;
    if constexpr (FLUX == PSA_FLUX_RUSANOV) sc.sR[tid + 1] = gF * duR;
  }
  __syncthreads();

  // ---- contributions of the cell to c - 2 .. c + 2
  if (tid >= 1 && tid <= B - 2) {
    const T cL = sc.cL[tid];
    T P[5];
    weno_cell_scatter(c, cR, cL, LEARNED && regime != 0, P);
    if constexpr (LEARNED) {
      if (regime == 2) {
#pragma unroll
        for (int r = 0; r < 5; ++r) P[r] += fma(cR, gR[r], cL * gL[r]);
      }
    }
    if constexpr (FLUX == PSA_FLUX_RUSANOV) P[2] += sL + sc.sR[tid];
#pragma unroll
    for (int r = 0; r < 5; ++r) sc.P[r][tid] = P[r];
  }
  __syncthreads();

  // ---- gather for output cell Z + tid (local computing index q)
  T gsum = T(0);
  if (tid < B - 6) {
    const int q = tid + 3;
#pragma unroll
    for (int r = 0; r < 5; ++r) gsum += sc.P[r][q + 2 - r];
  }
  return gsum;
}

// The reverse stage combinations from mu (the cotangent the stage received)
// and the gathered JL^T mu.
template <typename T, int RSTAGE>
__device__ __forceinline__ T vjp_value(T mu, T gsum, T dt, T lam, T lamk2) {
  if constexpr (RSTAGE == 0) {
    return gsum;
  } else if constexpr (RSTAGE == 3) {
    return T(2.0 / 3.0) * (mu + dt * gsum);
  } else if constexpr (RSTAGE == 2) {
    return T(1.0 / 4.0) * (mu + dt * gsum);
  } else {
    return (T(1.0 / 3.0) * lam + T(3.0 / 4.0) * lamk2) + (mu + dt * gsum);
  }
}

// RSTAGE 0: out = JL(state)^T mu; 3, 2, 1: the reverse stages above, with
// mu = l, lk2, lk1 respectively.
template <typename T, int FLUX, int RSTAGE, bool LEARNED = false>
__global__ __launch_bounds__(kVjpBlock) void k_stage_vjp(VjpArgs<T> p) {
  constexpr int B = kVjpBlock;
  __shared__ T s_u[B + 4];   // cells S - 5 ..
  __shared__ T s_mu[B + 1];  // cells S - 3 ..
  __shared__ VjpScratch<T, LEARNED> sc;

  const int tid = threadIdx.x;
  const int64_t n = p.n;
  const int g = p.g;
  const int64_t S = g + static_cast<int64_t>(blockIdx.x) * kVjpOut;

  if constexpr (FLUX == PSA_FLUX_LAX_FRIEDRICHS) {
    // the speed k_lf_alpha left in the output's first ghost entry (the
    // ghosts are cleared by k_lf_speed_vjp after this launch)
    p.alpha = p.out[0];
  } else if (blockIdx.x == 0 && tid < g) {
    // ghost entries of a cotangent are zero
    p.out[tid] = T(0);
    p.out[p.m - g + tid] = T(0);
  }

  if constexpr (LEARNED) vjp_net_load(sc.net, p.mlp);
  const PeriodicSpan cu(S - 5, n, g), cm(S - 3, n, g);
  for (int j = tid; j < B + 4; j += B) s_u[j] = cu.load(p.state, j);
  for (int j = tid; j < B + 1; j += B) s_mu[j] = cm.load(p.mu, j);
  __syncthreads();

  const T gsum = vjp_block<T, FLUX, LEARNED>(p, s_u, s_mu, sc);
  if (tid < kVjpOut) {
    const int64_t j = S + tid;
    if (j < p.m - g) {
      const T dt = RSTAGE == 0 ? T(0) : *p.dt_ptr;
      const T lam = RSTAGE == 1 ? p.lam[j] : T(0);
      const T lamk2 = RSTAGE == 1 ? p.lamk2[j] : T(0);
      p.out[j] = vjp_value<T, RSTAGE>(s_mu[tid + 3], gsum, dt, lam, lamk2);
    }
  }
}

// Arguments of the fused reverse steps.
template <typename T>
struct StepVjpArgs {
  VjpArgs<T> v;     // eps4, inv_dx, vconst, dt_ptr, m, n, g
  const T *x;       // the input state of the last step (the first one reversed)
  const T *k1;      // its stage states
  const T *k2;
  const T *lam;     // cotangent of that step's output
  T *out;           // cotangent of the input of the first step
  int64_t stride;   // from a step's states back to those of the step before
  int64_t bstride;  // a batch: instance blockIdx.y at offset blockIdx.y *
                    //   bstride of every array, its dt at dt_ptr[blockIdx.y]
  int nsub;         // steps reversed by the launch
};

// Waves per SIMD the registers of the plain reverse step are kept within.
#ifndef PSA_VJP_WAVES
#define PSA_VJP_WAVES 5
#endif

// Output cells per workgroup of nsub reverse steps.
constexpr int step_vjp_out(int nsub) { return kVjpBlock - 18 * nsub; }

// nsub reverse steps in one pass: a workgroup loads k2, k1, x and the incoming
// cotangent with halos of 11, 8, 5 and 9 cells around its window and runs
// reverse stages 3, 2 and 1 in LDS (vjp_block each). With the window's first
// cell S: lk2 is exact on [S - 6, S + B - 12), lk1 on [S - 3, S + B - 15), the
// step's cotangent on [S, S + B - 18); it is the next step's incoming
// cotangent, whose window starts 9 cells further in, so every step leaves 18
// cells fewer and the neighbouring workgroups recompute the margins. The same
// arithmetic as k_stage_vjp, and the same bits whatever nsub.
//
// One step per launch is mostly launch, load and drain at the size of a single
// gradient (N = 16384: 6.3 us a step, 3.1 of them the three stages), on a device
// that is nearly idle; several share that cost, and the next step's states are loaded while this
// one computes.
// MANY: more than one step (the registers of the states in flight, 90 instead
// of 66, would cost a batch a workgroup per CU).
template <typename T, int FLUX, bool LEARNED, bool MANY>
__global__ __launch_bounds__(kVjpBlock)
__attribute__((amdgpu_waves_per_eu(LEARNED ? (MANY ? 2 : 3) : PSA_VJP_WAVES))) void k_step_vjp(
    StepVjpArgs<T> a) {
  constexpr int B = kVjpBlock;
  __shared__ T sK2[B + 4], sK1[B + 4], sX[B + 4];
  __shared__ T sLam[B + 4];  // cells S - 9 ..
  __shared__ VjpScratch<T, LEARNED> sc;
  // lk2 (cells S - 6 ..) takes k2's buffer and lk1 (cells S - 3 ..) k1's:
  // each is written once the reverse stage that reads that state has
  // returned, and vjp_block reads its state only before its second barrier
  T *const sLk2 = sK2;
  T *const sLk1 = sK1;
  const VjpArgs<T> &p = a.v;
  const int tid = threadIdx.x;
  const int64_t n = p.n;
  const int g = p.g;
  const int nsub = MANY ? a.nsub : 1;
  const int nout = step_vjp_out(nsub);
  // the workgroup's output cells start at A, the first step's window at S
  const int64_t A = g + static_cast<int64_t>(blockIdx.x) * nout;
  const int64_t S = A - 9 * (nsub - 1);
  const int64_t off = static_cast<int64_t>(blockIdx.y) * a.bstride;
  const T dt = p.dt_ptr[blockIdx.y];
  const T *xk2 = a.k2 + off;
  const T *xk1 = a.k1 + off;
  const T *xx = a.x + off;
  T *xout = a.out + off;

  if (blockIdx.x == 0 && tid < g) {
    xout[tid] = T(0);
    xout[p.m - g + tid] = T(0);
  }
  if constexpr (LEARNED) vjp_net_load(sc.net, p.mlp);
  // cells S - 11 + j of the periodic array
  const PeriodicSpan span(S - 11, n, g);
  const bool more = tid < 4;
  {
    const T *xlam = a.lam + off;
    for (int j = tid; j < B + 4; j += B) {
      sK2[j] = span.load(xk2, j);
      sK1[j] = span.load(xk1, j + 3);
      sX[j] = span.load(xx, j + 6);
      sLam[j] = span.load(xlam, j + 2);
    }
  }
  __syncthreads();

  for (int s = 0; s < nsub; ++s) {
    // the next step's states (window 9 cells further in)
    const bool next = MANY && s + 1 < nsub;
    T n2 = T(0), n1 = T(0), nx = T(0), e2 = T(0), e1 = T(0), ex = T(0);
    if (next) {
      const int64_t back = (s + 1) * a.stride;
      const int j = tid + 9 * (s + 1);
      n2 = span.load(xk2 - back, j);
      n1 = span.load(xk1 - back, j + 3);
      nx = span.load(xx - back, j + 6);
      if (more) {
        e2 = span.load(xk2 - back, j + B);
        e1 = span.load(xk1 - back, j + B + 3);
        ex = span.load(xx - back, j + B + 6);
      }
    }
    // reverse stage 3 on the output cells S - 6 + t: lk2 (with zeros in the
    // entries past the exact cotangents, read only for cells outside the exact
    // ranges: finite values)
    T gsum = vjp_block<T, FLUX, LEARNED>(p, sK2, sLam, sc);
    sLk2[tid] = tid < B - 6 ? vjp_value<T, 3>(sLam[tid + 3], gsum, dt, T(0), T(0)) : T(0);
    if (tid == 0) sLk2[B] = T(0);
    __syncthreads();
    // reverse stage 2 on S - 3 + t: lk1
    gsum = vjp_block<T, FLUX, LEARNED>(p, sK1, sLk2, sc);
    sLk1[tid] = tid < B - 6 ? vjp_value<T, 2>(sLk2[tid + 3], gsum, dt, T(0), T(0)) : T(0);
    if (tid == 0) sLk1[B] = T(0);
    __syncthreads();
    // reverse stage 1 on S + t: the cotangent of the step input
    gsum = vjp_block<T, FLUX, LEARNED>(p, sX, sLk1, sc);
    const T lam = tid < B - 18 ? vjp_value<T, 1>(sLk1[tid + 3], gsum, dt, sLam[tid + 9],
                                                 sLk2[tid + 6])
                               : T(0);
    if (!next) {
      const int64_t j = A + tid;
      if (tid < nout && j < p.m - g) xout[j] = lam;
      break;
    }
    __syncthreads();
    sLam[tid] = lam;
    sK2[tid] = n2;
    sK1[tid] = n1;
    sX[tid] = nx;
    if (more) {
      sLam[B + tid] = T(0);
      sK2[B + tid] = e2;
      sK1[B + tid] = e1;
      sX[B + tid] = ex;
    }
    __syncthreads();
  }
}

template <typename T>
__global__ void k_zero_ghosts(T *u, int64_t m, int g, int64_t ld) {
  const int t = threadIdx.x;
  T *v = u + static_cast<int64_t>(blockIdx.x) * ld;
  if (t < g) {
    v[t] = T(0);
    v[m - g + t] = T(0);
  }
}

// ---------------------------------------------------------------------------
// Lax-Friedrichs: the global speed alpha = max |state| over the ghost-filled
// array (scalar.py:276-277) couples every face to the cells where |state|
// is largest. One workgroup each: k_lf_alpha puts alpha into out[0] (a
// ghost entry) for k_stage_vjp, which differentiates the faces at fixed
// alpha; k_lf_speed_vjp then adds the derivative through alpha, G =
// sum over the faces of gF dF/dalpha, dF/dalpha = -(ul - ur) / 2, shared by
// the entries of the ghost-filled array where |state| = alpha (jax's max:
// ties share equally; d|x|/dx = sign(x)), mapped to their cells through the
// periodic fill, and clears the ghost entries.

constexpr int kLfBlock = 256;

template <typename T>
__device__ __forceinline__ T lf_block_sum(T v, T *s_red) {
  const int tid = threadIdx.x;
  s_red[tid] = v;
  __syncthreads();
  for (int w = kLfBlock / 2; w > 0; w >>= 1) {
    if (tid < w) s_red[tid] = s_red[tid] + s_red[tid + w];
    __syncthreads();
  }
  const T r = s_red[0];
  __syncthreads();
  return r;
}

template <typename T>
__global__ __launch_bounds__(kLfBlock) void k_lf_alpha(VjpArgs<T> p) {
  __shared__ T s_red[kLfBlock];
  const int tid = threadIdx.x;
  T mx = T(0);
  bool nan = false;
  for (int64_t c = p.g + tid; c < p.m - p.g; c += kLfBlock) {
    const T v = p.state[c];
    mx = fmax(mx, fabs(v));
    nan |= isnan(v);
  }
  s_red[tid] = nan ? T(NAN) : mx;
  __syncthreads();
  for (int w = kLfBlock / 2; w > 0; w >>= 1) {
    if (tid < w) {
      const T a = s_red[tid], b = s_red[tid + w];
      s_red[tid] = (isnan(a) || isnan(b)) ? T(NAN) : fmax(a, b);
    }
    __syncthreads();
  }
  if (tid == 0) p.out[0] = s_red[0];
}

template <typename T, int RSTAGE>
__global__ __launch_bounds__(kLfBlock) void k_lf_speed_vjp(VjpArgs<T> p) {
  __shared__ T s_red[kLfBlock];
  const int tid = threadIdx.x;
  const int64_t n = p.n, m = p.m;
  const int g = p.g;
  const T alpha = p.out[0];
  // G over the n faces of the periodic ring (face j between cells j - 1, j)
  T acc = T(0);
  for (int64_t j = g + tid; j < m - g; j += kLfBlock) {
    const PeriodicSpan span(j - 3, n, g);
    T v[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) v[k] = span.load(p.state, k);
    CellStates<T> c;
    T urL, ulR, unused;
    weno_cell_states(v, p.eps4, c, unused, urL);
    weno_cell_states(v + 1, p.eps4, c, ulR, unused);
    const T gF = (span.load(p.mu, 3) - span.load(p.mu, 2)) * p.inv_dx;
    acc += gF * (T(-0.5) * (ulR - urL));
  }
  const T G = lf_block_sum(acc, s_red);
  // entries of the ghost-filled array that hold cell c: c itself, the left
  // ghost c - n for cells n .. n + g - 1 and the right ghost c + n for cells
  // g .. 2g - 1
  auto mult = [&](int64_t c) {
    return 1 + ((c >= n && c < n + g) ? 1 : 0) + ((c >= g && c < 2 * g) ? 1 : 0);
  };
  T cnt = T(0);
  for (int64_t c = g + tid; c < m - g; c += kLfBlock)
    if (fabs(p.state[c]) == alpha) cnt += T(mult(c));
  const T count = lf_block_sum(cnt, s_red);
  T coef = T(1);
  if constexpr (RSTAGE == 3) {
    coef = T(2.0 / 3.0) * *p.dt_ptr;
  } else if constexpr (RSTAGE == 2) {
    coef = T(1.0 / 4.0) * *p.dt_ptr;
  } else if constexpr (RSTAGE == 1) {
    coef = *p.dt_ptr;
  }
  if (count > T(0)) {
    const T share = coef * G / count;
    for (int64_t c = g + tid; c < m - g; c += kLfBlock) {
      const T v = p.state[c];
      if (fabs(v) == alpha) p.out[c] += share * T(mult(c)) * sgn(v);
    }
  }
  // the ghost entries (out[0] carried alpha; every thread read it above)
  if (tid < g) {
    p.out[tid] = T(0);
    p.out[m - g + tid] = T(0);
  }
}

template <typename T, int FLUX, bool LEARNED = false>
int launch_vjp_flux(int rstage, const VjpArgs<T> &a, hipStream_t s) {
  const unsigned int blocks =
      static_cast<unsigned int>((a.n + kVjpOut - 1) / kVjpOut);
  switch (rstage) {
    case 0:
      hipLaunchKernelGGL((k_stage_vjp<T, FLUX, 0, LEARNED>), dim3(blocks),
                         dim3(kVjpBlock), 0, s, a);
      break;
    case 1:
      hipLaunchKernelGGL((k_stage_vjp<T, FLUX, 1, LEARNED>), dim3(blocks),
                         dim3(kVjpBlock), 0, s, a);
      break;
    case 2:
      hipLaunchKernelGGL((k_stage_vjp<T, FLUX, 2, LEARNED>), dim3(blocks),
                         dim3(kVjpBlock), 0, s, a);
      break;
    default:
      hipLaunchKernelGGL((k_stage_vjp<T, FLUX, 3, LEARNED>), dim3(blocks),
                         dim3(kVjpBlock), 0, s, a);
      break;
  }
  return check_launch("stage vjp");
}

template <typename T>
int launch_vjp(const psa_solver_desc *d, int rstage, const void *state,
               const void *mu, const void *lam, const void *lamk2, void *out,
               const void *dt, hipStream_t s) {
  VjpArgs<T> a{};
  a.state = static_cast<const T *>(state);
  a.mu = static_cast<const T *>(mu);
  a.lam = static_cast<const T *>(lam);
  a.lamk2 = static_cast<const T *>(lamk2);
  a.out = static_cast<T *>(out);
  a.dt_ptr = static_cast<const T *>(dt);
  a.n = d->n;
  a.g = d->g;
  a.m = d->n + 2 * static_cast<int64_t>(d->g);
  a.inv_dx = T(1) / static_cast<T>(d->dx);
  a.eps = static_cast<T>(d->eps);
  a.vconst = static_cast<T>(d->velocity_const);
  a.mlp = d->mlp;
  a.eps4 = T(4) * a.eps;
  a.tau = static_cast<T>(d->mlp_tau);
  a.sigma = static_cast<T>(d->mlp_sigma);
  if (d->mlp != nullptr) {
    if (d->flux == PSA_FLUX_RUSANOV)
      return launch_vjp_flux<T, PSA_FLUX_RUSANOV, true>(rstage, a, s);
    if (d->flux == PSA_FLUX_ENGQUIST_OSHER)
      return launch_vjp_flux<T, PSA_FLUX_ENGQUIST_OSHER, true>(rstage, a, s);
    return launch_vjp_flux<T, PSA_FLUX_BURGERS_UPWIND, true>(rstage, a, s);
  }
  if (d->flux == PSA_FLUX_LAX_FRIEDRICHS) {
    hipLaunchKernelGGL(k_lf_alpha<T>, dim3(1), dim3(kLfBlock), 0, s, a);
    int st = check_launch("speed of the stage");
    if (st != PSA_OK) return st;
    st = launch_vjp_flux<T, PSA_FLUX_LAX_FRIEDRICHS>(rstage, a, s);
    if (st != PSA_OK) return st;
    switch (rstage) {
      case 0:
        hipLaunchKernelGGL((k_lf_speed_vjp<T, 0>), dim3(1), dim3(kLfBlock), 0, s, a);
        break;
      case 1:
        hipLaunchKernelGGL((k_lf_speed_vjp<T, 1>), dim3(1), dim3(kLfBlock), 0, s, a);
        break;
      case 2:
        hipLaunchKernelGGL((k_lf_speed_vjp<T, 2>), dim3(1), dim3(kLfBlock), 0, s, a);
        break;
      default:
        hipLaunchKernelGGL((k_lf_speed_vjp<T, 3>), dim3(1), dim3(kLfBlock), 0, s, a);
        break;
    }
    return check_launch("speed vjp");
  }
  if (d->flux == PSA_FLUX_RUSANOV)
    return launch_vjp_flux<T, PSA_FLUX_RUSANOV>(rstage, a, s);
  if (d->flux == PSA_FLUX_BURGERS_UPWIND)
    return launch_vjp_flux<T, PSA_FLUX_BURGERS_UPWIND>(rstage, a, s);
  if (d->flux == PSA_FLUX_ENGQUIST_OSHER)
    return launch_vjp_flux<T, PSA_FLUX_ENGQUIST_OSHER>(rstage, a, s);
  return launch_vjp_flux<T, PSA_FLUX_ADVECTION_UPWIND>(rstage, a, s);
}

// Reverse steps that a launch best takes. Measured (FP64, Rusanov; us a step
// with 1 step per launch and with the chosen number, before the six operations
// that keep the weights' gradients exact beside a jump, 2 to 3% more since): one
// instance of 256 cells 5.33 -> 3.41, of 16384 6.31 -> 3.41, of 65536 7.19 -> 4.48;
// 16 instances of 16384 11.6 -> 9.5.
int reverse_steps_per_launch(const psa_solver_desc *d, long long batch) {
  return best_steps(StepCost{3.3, 2.0, 1.0}, kVjpMostSteps, [&](int k) {
    const int nout = step_vjp_out(k);
    return (d->n + nout - 1) / nout * batch;
  });
}

template <typename T, bool MANY>
void launch_step_vjp_flux(const psa_solver_desc *d, const StepVjpArgs<T> &a, dim3 grid,
                          hipStream_t s) {
  const dim3 block(kVjpBlock);
  if (d->mlp != nullptr) {
    if (d->flux == PSA_FLUX_RUSANOV) {
      hipLaunchKernelGGL((k_step_vjp<T, PSA_FLUX_RUSANOV, true, MANY>), grid, block, 0, s, a);
    } else if (d->flux == PSA_FLUX_ENGQUIST_OSHER) {
      hipLaunchKernelGGL((k_step_vjp<T, PSA_FLUX_ENGQUIST_OSHER, true, MANY>), grid, block, 0,
                         s, a);
    } else {
      hipLaunchKernelGGL((k_step_vjp<T, PSA_FLUX_BURGERS_UPWIND, true, MANY>), grid, block, 0,
                         s, a);
    }
  } else if (d->flux == PSA_FLUX_RUSANOV) {
    hipLaunchKernelGGL((k_step_vjp<T, PSA_FLUX_RUSANOV, false, MANY>), grid, block, 0, s, a);
  } else if (d->flux == PSA_FLUX_BURGERS_UPWIND) {
    hipLaunchKernelGGL((k_step_vjp<T, PSA_FLUX_BURGERS_UPWIND, false, MANY>), grid, block, 0,
                       s, a);
  } else if (d->flux == PSA_FLUX_ENGQUIST_OSHER) {
    hipLaunchKernelGGL((k_step_vjp<T, PSA_FLUX_ENGQUIST_OSHER, false, MANY>), grid, block, 0,
                       s, a);
  } else {
    hipLaunchKernelGGL((k_step_vjp<T, PSA_FLUX_ADVECTION_UPWIND, false, MANY>), grid, block, 0,
                       s, a);
  }
}

// nsub reverse steps as one launch (k_step_vjp): x, k1, k2 of the last of the
// steps, those of the step before `stride` elements before them.
template <typename T>
int launch_step_vjp(const psa_solver_desc *d, const void *x, const void *k1,
                    const void *k2, const void *lam, void *out, const void *dt,
                    long long nsub, int64_t stride, hipStream_t s, long long batch,
                    int64_t ld) {
  StepVjpArgs<T> a{};
  a.bstride = ld;
  a.stride = stride;
  a.nsub = static_cast<int>(nsub);
  a.v.mlp = d->mlp;
  a.v.eps4 = T(4) * static_cast<T>(d->eps);
  a.v.tau = static_cast<T>(d->mlp_tau);
  a.v.sigma = static_cast<T>(d->mlp_sigma);
  a.v.dt_ptr = static_cast<const T *>(dt);
  a.v.n = d->n;
  a.v.g = d->g;
  a.v.m = d->n + 2 * static_cast<int64_t>(d->g);
  a.v.inv_dx = T(1) / static_cast<T>(d->dx);
  a.v.eps = static_cast<T>(d->eps);
  a.v.vconst = static_cast<T>(d->velocity_const);
  a.x = static_cast<const T *>(x);
  a.k1 = static_cast<const T *>(k1);
  a.k2 = static_cast<const T *>(k2);
  a.lam = static_cast<const T *>(lam);
  a.out = static_cast<T *>(out);
  const int nout = step_vjp_out(a.nsub);
  const dim3 grid(static_cast<unsigned int>((d->n + nout - 1) / nout),
                  static_cast<unsigned int>(batch));
  if (a.nsub > 1) {
    launch_step_vjp_flux<T, true>(d, a, grid, s);
  } else {
    launch_step_vjp_flux<T, false>(d, a, grid, s);
  }
  return check_launch("step vjp");
}

int check_vjp_desc(const psa_solver_desc *d) {
  if (d == nullptr) return set_error(PSA_ERR_INVALID_ARGUMENT, "null desc");
  if (d->dtype != PSA_FLOAT64 && d->dtype != PSA_FLOAT32)
    return set_error(PSA_ERR_NOT_IMPLEMENTED, "unsupported dtype");
  if (d->rec != PSA_REC_WENOJS53)
    return set_error(PSA_ERR_NOT_IMPLEMENTED,
                     "the adjoint supports the WENO-JS5 reconstruction only");
  if (d->bc != PSA_BC_PERIODIC)
    return set_error(PSA_ERR_NOT_IMPLEMENTED, "the adjoint is periodic");
  if (d->g < 3 || d->n < d->g)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "bad grid size");
  if (d->flux < 0 || d->flux > PSA_FLUX_LAX_FRIEDRICHS)
    return set_error(PSA_ERR_NOT_IMPLEMENTED, "unsupported flux");
  if ((d->flux == PSA_FLUX_RUSANOV || d->flux == PSA_FLUX_LAX_FRIEDRICHS) &&
      d->nu != nullptr)
    return set_error(PSA_ERR_NOT_IMPLEMENTED,
                     "the adjoint supports the Rusanov and Lax-Friedrichs fluxes "
                     "with alpha = 1");
  if (d->flux == PSA_FLUX_LAX_FRIEDRICHS && d->mlp != nullptr)
    return set_error(PSA_ERR_NOT_IMPLEMENTED,
                     "the adjoint of learned weights takes Rusanov, Godunov and "
                     "Engquist-Osher");
  if (d->flux == PSA_FLUX_ADVECTION_UPWIND && !d->velocity_is_const)
    return set_error(PSA_ERR_NOT_IMPLEMENTED,
                     "the adjoint supports advection with a constant velocity");
  if (d->mlp != nullptr && d->flux == PSA_FLUX_ADVECTION_UPWIND)
    return set_error(PSA_ERR_NOT_IMPLEMENTED,
                     "the adjoint of learned weights takes the Burgers fluxes");
  if (d->mlp != nullptr && (!(d->mlp_tau >= 0.0) || !(d->mlp_sigma >= 0.0)))
    return set_error(PSA_ERR_INVALID_ARGUMENT, "mlp_tau and mlp_sigma must be >= 0");
  if (!(d->dx > 0.0))
    return set_error(PSA_ERR_INVALID_ARGUMENT, "dx must be positive");
  return PSA_OK;
}

size_t elem_size(const psa_solver_desc *d) {
  return d->dtype == PSA_FLOAT64 ? sizeof(double) : sizeof(float);
}

int copy_async(void *dst, const void *src, size_t bytes, hipStream_t s) {
  hipError_t err = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, s);
  if (err != hipSuccess) return set_error(PSA_ERR_HIP, hipGetErrorString(err));
  return PSA_OK;
}

struct AdjointLayout {
  long long ncp;     // checkpoints at steps 0, every, 2 every, ...
  long long nwin;    // arrays of the recompute window
  size_t array_bytes;
  size_t bytes;
};

// batch instances at a stride of ld elements per array (ld = m for one)
AdjointLayout adjoint_layout(const psa_solver_desc *d, long long nsteps,
                             int every, long long batch = 1, int64_t ld = 0) {
  AdjointLayout L{};
  const size_t m = static_cast<size_t>(d->n + 2 * static_cast<int64_t>(d->g));
  const size_t cells = batch > 1 ? static_cast<size_t>(batch) * static_cast<size_t>(ld) : m;
  L.array_bytes = ((cells * elem_size(d) + 255) / 256) * 256;
  L.ncp = nsteps / every + 1;
  L.nwin = 3LL * every;
  // checkpoints, window (x, k1, k2 per step), running state, 4 cotangents,
  // and 256 bytes for the Lax-Friedrichs stage speed
  L.bytes = static_cast<size_t>(L.ncp + L.nwin + 1 + 4) * L.array_bytes + 256;
  return L;
}

// The device scalar of the Lax-Friedrichs stage speed in the workspace.
void *lf_speed_slot(void *workspace, const AdjointLayout &L) {
  return static_cast<char *>(workspace) + (L.bytes - 256);
}

}  // namespace
}  // namespace psa

// defined in forward.hip and reductions.hip
extern "C" int psa_ssprk33_stage(const psa_solver_desc *desc, int stage,
                                 const void *un, const void *uk, void *out,
                                 void *control, const void *dt, void *stream);
extern "C" int psa_max_abs_interior(int dtype, const void *u, void *out, int64_t m,
                                    int g, void *stream);

using namespace psa;

namespace {

// One fixed-dt stage (psa_ssprk33_stage without a control block); for
// Lax-Friedrichs the flux speed max|uk| of the stage input first goes to the
// device scalar speed (scalar.py:276-277: the interior maximum, the ghosts
// being images).
int forward_stage(const psa_solver_desc *d, int stage, const void *un, const void *uk,
                  void *out, const void *dt, void *speed, void *stream) {
  if (d->flux != PSA_FLUX_LAX_FRIEDRICHS)
    return psa_ssprk33_stage(d, stage, un, uk, out, nullptr, dt, stream);
  const int64_t m = d->n + 2 * static_cast<int64_t>(d->g);
  const int st = psa_max_abs_interior(d->dtype, uk, speed, m, d->g, stream);
  if (st != PSA_OK) return st;
  psa_solver_desc dl = *d;
  dl.velocity = speed;
  return psa_ssprk33_stage(&dl, stage, un, uk, out, nullptr, dt, stream);
}

}  // namespace

extern "C" {

int psa_ssprk33_stage_vjp(const psa_solver_desc *desc, int stage,
                          const void *state, const void *mu, const void *lam,
                          const void *lam_k2, void *out, const void *dt,
                          void *stream) {
  int st = check_vjp_desc(desc);
  if (st != PSA_OK) return st;
  if (stage < 0 || stage > 3)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "stage must be 0..3");
  if (state == nullptr || mu == nullptr || out == nullptr ||
      (stage > 0 && dt == nullptr) ||
      (stage == 1 && (lam == nullptr || lam_k2 == nullptr)))
    return set_error(PSA_ERR_INVALID_ARGUMENT, "null pointer");
  if (out == mu || out == state || (stage == 1 && (out == lam || out == lam_k2)))
    return set_error(PSA_ERR_INVALID_ARGUMENT,
                     "the output must not alias an input");
  auto s = static_cast<hipStream_t>(stream);
  if (desc->dtype == PSA_FLOAT64)
    return launch_vjp<double>(desc, stage, state, mu, lam, lam_k2, out, dt, s);
  return launch_vjp<float>(desc, stage, state, mu, lam, lam_k2, out, dt, s);
}

int psa_ssprk33_step_vjp(const psa_solver_desc *desc, const void *u,
                         const void *lam, void *lam_out, void *work,
                         size_t work_bytes, const void *dt, void *stream) {
  int st = check_vjp_desc(desc);
  if (st != PSA_OK) return st;
  if (u == nullptr || lam == nullptr || lam_out == nullptr || work == nullptr ||
      dt == nullptr)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "null pointer");
  const size_t m = static_cast<size_t>(desc->n + 2 * static_cast<int64_t>(desc->g));
  const size_t ab = ((m * elem_size(desc) + 255) / 256) * 256;
  if (work_bytes < 4 * ab)
    return set_error(PSA_ERR_WORKSPACE, "step vjp needs 4 arrays of workspace");
  if (lam_out == lam || lam_out == u)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "lam_out must not alias");
  char *w = static_cast<char *>(work);
  void *k1 = w, *k2 = w + ab, *lk2 = w + 2 * ab, *lk1 = w + 3 * ab;
  // recompute the stages of the forward step (a Lax-Friedrichs stage speed
  // in lk1's storage, which the reverse stages write later)
  st = forward_stage(desc, 1, u, u, k1, dt, lk1, stream);
  if (st != PSA_OK) return st;
  st = forward_stage(desc, 2, u, k1, k2, dt, lk1, stream);
  if (st != PSA_OK) return st;

  st = psa_ssprk33_stage_vjp(desc, 3, k2, lam, nullptr, nullptr, lk2, dt, stream);
  if (st != PSA_OK) return st;
  st = psa_ssprk33_stage_vjp(desc, 2, k1, lk2, nullptr, nullptr, lk1, dt, stream);
  if (st != PSA_OK) return st;
  return psa_ssprk33_stage_vjp(desc, 1, u, lk1, lam, lk2, lam_out, dt, stream);
}

}  // extern "C"

namespace {

// The batch arguments: batch >= 1 instances at ld >= m elements apart (ld a
// multiple of 16 bytes), whole-step kernels only when batch > 1.
int check_batch(const psa_solver_desc *d, long long batch, long long ld) {
  const int64_t m = d->n + 2 * static_cast<int64_t>(d->g);
  if (batch < 1 || batch > 65535)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "batch must be in [1, 65535]");
  if (batch > 1 && (ld < m || (ld * static_cast<long long>(elem_size(d))) % 16 != 0))
    return set_error(PSA_ERR_INVALID_ARGUMENT,
                     "ld must be >= m and a multiple of 16 bytes");
  return PSA_OK;
}

// With one window over the whole horizon the forward pass keeps the window's
// states itself (the window's 3 every arrays hold all of them, X(nsteps)
// being at most the running-state array X(every)).
bool keeps_window(long long nsteps, int every) { return nsteps > 0 && every >= nsteps; }

// Whole steps the next launch takes of the `left` ones; 0 where the whole-step
// kernels do not apply.
long long steps_now(const psa_solver_desc *d, long long batch, long long left) {
  const long long k = fixed_steps_per_launch(d, batch);
  return k < left ? k : left;
}

// The step of the first checkpoint after `step`, or the last step.
long long checkpoint_after(long long step, int every, long long nsteps) {
  const long long next = (step / every + 1) * every;
  return next < nsteps ? next : nsteps;
}

int batch_needs_steps() {
  return set_error(PSA_ERR_NOT_IMPLEMENTED,
                   "a batch runs on the whole-step kernel (default or step "
                   "schedule, tiles 256 x 4 or 256 x 2, not Lax-Friedrichs)");
}

int forward_checkpointed(const psa_solver_desc *desc, long long batch, int64_t ld,
                         const void *u0, void *u_final, long long nsteps,
                         const void *dt, int every, void *workspace,
                         size_t workspace_bytes, hipStream_t s) {
  int st = check_vjp_desc(desc);
  if (st != PSA_OK) return st;
  st = check_batch(desc, batch, ld);
  if (st != PSA_OK) return st;
  if (u0 == nullptr || u_final == nullptr || dt == nullptr ||
      workspace == nullptr || nsteps < 0 || every <= 0)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "bad arguments");
  const AdjointLayout L = adjoint_layout(desc, nsteps, every, batch, ld);
  if (workspace_bytes < L.bytes)
    return set_error(PSA_ERR_WORKSPACE, "adjoint workspace too small");
  const size_t m = static_cast<size_t>(desc->n + 2 * static_cast<int64_t>(desc->g));
  const size_t bytes =
      (batch > 1 ? static_cast<size_t>(batch) * static_cast<size_t>(ld) : m) *
      elem_size(desc);
  char *base = static_cast<char *>(workspace);
  auto cp = [&](long long k) { return base + k * L.array_bytes; };
  char *win = cp(L.ncp);
  const int64_t step_stride = static_cast<int64_t>(3 * L.array_bytes / elem_size(desc));
  char *cur = win + L.nwin * L.array_bytes;
  void *k1 = win, *k2 = win + L.array_bytes;

  st = copy_async(cp(0), u0, bytes, s);
  if (st != PSA_OK) return st;
  if (keeps_window(nsteps, every)) {
    // one window over the whole horizon: keep every step's states (x, k1,
    // k2) in it now, so that the reverse sweep recomputes nothing
    auto X = [&](long long i) { return win + (3 * i) * L.array_bytes; };
    auto K1 = [&](long long i) { return win + (3 * i + 1) * L.array_bytes; };
    auto K2 = [&](long long i) { return win + (3 * i + 2) * L.array_bytes; };
    st = copy_async(X(0), u0, bytes, s);
    if (st != PSA_OK) return st;
    for (long long i = 0; i < nsteps;) {
      const long long k = steps_now(desc, batch, nsteps - i);
      if (k > 0) {
        st = steps_fixed_dt(desc, X(i), X(i + 1), K1(i), K2(i), k, step_stride, dt, s, batch,
                            ld);
        if (st != PSA_OK) return st;
        i += k;
        continue;
      }
      if (batch > 1) return batch_needs_steps();
      void *speed = lf_speed_slot(workspace, L);
      st = forward_stage(desc, 1, X(i), X(i), K1(i), dt, speed, s);
      if (st != PSA_OK) return st;
      st = forward_stage(desc, 2, X(i), K1(i), K2(i), dt, speed, s);
      if (st != PSA_OK) return st;
      st = forward_stage(desc, 3, X(i), K2(i), X(i + 1), dt, speed, s);
      if (st != PSA_OK) return st;
      ++i;
    }
    if (nsteps % every == 0) {
      st = copy_async(cp(1), X(nsteps), bytes, s);
      if (st != PSA_OK) return st;
    }
    return copy_async(u_final, X(nsteps), bytes, s);
  }
  st = copy_async(cur, u0, bytes, s);
  if (st != PSA_OK) return st;
  // whole steps, the state alternating between cur and the window's first
  // array, where the whole-step kernel applies
  char *alt = win;
  for (long long step = 0; step < nsteps;) {
    // (up to the next checkpoint)
    const long long k = steps_now(desc, batch, checkpoint_after(step, every, nsteps) - step);
    if (k > 0) {
      st = steps_fixed_dt(desc, cur, alt, nullptr, nullptr, k, 0, dt, s, batch, ld);
      if (st != PSA_OK) return st;
      char *tmp = cur;
      cur = alt;
      alt = tmp;
      step += k;
      if (step % every == 0) {
        st = copy_async(cp(step / every), cur, bytes, s);
        if (st != PSA_OK) return st;
      }
      continue;
    }
    if (batch > 1) return batch_needs_steps();
    void *speed = lf_speed_slot(workspace, L);
    st = forward_stage(desc, 1, cur, cur, k1, dt, speed, s);
    if (st != PSA_OK) return st;
    st = forward_stage(desc, 2, cur, k1, k2, dt, speed, s);
    if (st != PSA_OK) return st;
    st = forward_stage(desc, 3, cur, k2, cur, dt, speed, s);
    if (st != PSA_OK) return st;
    ++step;
    if (step % every == 0) {
      st = copy_async(cp(step / every), cur, bytes, s);
      if (st != PSA_OK) return st;
    }
  }
  return copy_async(u_final, cur, bytes, s);
}

int adjoint(const psa_solver_desc *desc, long long batch, int64_t ld, long long nsteps,
            const void *dt, int every, const void *lam_final, void *grad_u0,
            void *workspace, size_t workspace_bytes, hipStream_t s) {
  int st = check_vjp_desc(desc);
  if (st != PSA_OK) return st;
  st = check_batch(desc, batch, ld);
  if (st != PSA_OK) return st;
  if (lam_final == nullptr || grad_u0 == nullptr || dt == nullptr ||
      workspace == nullptr || nsteps < 0 || every <= 0)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "bad arguments");
  const AdjointLayout L = adjoint_layout(desc, nsteps, every, batch, ld);
  if (workspace_bytes < L.bytes)
    return set_error(PSA_ERR_WORKSPACE, "adjoint workspace too small");
  const size_t m = static_cast<size_t>(desc->n + 2 * static_cast<int64_t>(desc->g));
  const size_t bytes =
      (batch > 1 ? static_cast<size_t>(batch) * static_cast<size_t>(ld) : m) *
      elem_size(desc);
  char *base = static_cast<char *>(workspace);
  auto cp = [&](long long k) { return base + k * L.array_bytes; };
  char *win = cp(L.ncp);
  const int64_t step_stride = static_cast<int64_t>(3 * L.array_bytes / elem_size(desc));
  auto X = [&](long long i) { return win + (3 * i) * L.array_bytes; };
  auto K1 = [&](long long i) { return win + (3 * i + 1) * L.array_bytes; };
  auto K2 = [&](long long i) { return win + (3 * i + 2) * L.array_bytes; };
  char *lam_a = win + L.nwin * L.array_bytes + L.array_bytes;
  char *lam_b = lam_a + L.array_bytes;
  char *lk2 = lam_b + L.array_bytes;
  char *lk1 = lk2 + L.array_bytes;
  // (Lax-Friedrichs: the stage-wise reverse, whose global speed term needs a
  // reduction between the stages)
  if (desc->flux == PSA_FLUX_LAX_FRIEDRICHS && batch > 1)
    return set_error(PSA_ERR_NOT_IMPLEMENTED,
                     "the batched adjoint does not take Lax-Friedrichs");
  const bool fused_reverse =
      desc->flux != PSA_FLUX_LAX_FRIEDRICHS &&
      (batch > 1 || (desc->schedule != PSA_SCHEDULE_TILE &&
                     desc->schedule != PSA_SCHEDULE_PIPELINE));

  const long long reverse_most = reverse_steps_per_launch(desc, batch);

  st = copy_async(lam_a, lam_final, bytes, s);
  if (st != PSA_OK) return st;
  char *lam = lam_a, *lam_next = lam_b;
  const long long nwin = (nsteps + every - 1) / every;
  for (long long w = nwin - 1; w >= 0; --w) {
    const long long s0 = w * every;
    const long long s1 = (s0 + every < nsteps) ? s0 + every : nsteps;
    // recompute the window from its checkpoint, keeping every stage state
    // (kept by the forward pass already when it spans the horizon)
    const bool kept = keeps_window(nsteps, every);
    if (!kept) {
      st = copy_async(X(0), cp(w), bytes, s);
      if (st != PSA_OK) return st;
    }
    for (long long step = s0; step < s1 && !kept;) {
      const long long i = step - s0;
      // whole steps writing k1, k2 and the next state (X(every) is the
      // running-state array, free in this pass)
      const long long k = steps_now(desc, batch, s1 - step);
      if (k > 0) {
        st = steps_fixed_dt(desc, X(i), X(i + 1), K1(i), K2(i), k, step_stride, dt, s, batch,
                            ld);
        if (st != PSA_OK) return st;
        step += k;
        continue;
      }
      if (batch > 1) return batch_needs_steps();
      void *speed = lf_speed_slot(workspace, L);
      st = forward_stage(desc, 1, X(i), X(i), K1(i), dt, speed, s);
      if (st != PSA_OK) return st;
      st = forward_stage(desc, 2, X(i), K1(i), K2(i), dt, speed, s);
      if (st != PSA_OK) return st;
      if (step + 1 < s1) {
        st = forward_stage(desc, 3, X(i), K2(i), X(i + 1), dt, speed, s);
        if (st != PSA_OK) return st;
      }
      ++step;
    }
    // reverse sweep through the window
    for (long long step = s1 - 1; step >= s0; --step) {
      const long long i = step - s0;
      if (fused_reverse) {
        // the three reverse stages of this step and of some before it in one
        // launch
        const long long k = reverse_most < i + 1 ? reverse_most : i + 1;
        st = desc->dtype == PSA_FLOAT64
                 ? launch_step_vjp<double>(desc, X(i), K1(i), K2(i), lam, lam_next, dt, k,
                                           step_stride, s, batch, ld)
                 : launch_step_vjp<float>(desc, X(i), K1(i), K2(i), lam, lam_next, dt, k,
                                          step_stride, s, batch, ld);
        if (st != PSA_OK) return st;
        step -= k - 1;
        char *tmp = lam;
        lam = lam_next;
        lam_next = tmp;
        continue;
      }
      st = psa_ssprk33_stage_vjp(desc, 3, K2(i), lam, nullptr, nullptr, lk2, dt, s);
      if (st != PSA_OK) return st;
      st = psa_ssprk33_stage_vjp(desc, 2, K1(i), lk2, nullptr, nullptr, lk1, dt, s);
      if (st != PSA_OK) return st;
      st = psa_ssprk33_stage_vjp(desc, 1, X(i), lk1, lam, lk2, lam_next, dt, s);
      if (st != PSA_OK) return st;
      char *tmp = lam;
      lam = lam_next;
      lam_next = tmp;
    }
  }
  st = copy_async(grad_u0, lam, bytes, s);
  if (st != PSA_OK) return st;
  if (nsteps == 0) {
    // no step: the gradient is the incoming cotangent with zero ghosts
    const int64_t mm = static_cast<int64_t>(m);
    const dim3 grid(static_cast<unsigned int>(batch));
    if (desc->dtype == PSA_FLOAT64) {
      hipLaunchKernelGGL(k_zero_ghosts<double>, grid, dim3(64), 0, s,
                         static_cast<double *>(grad_u0), mm, desc->g, ld);
    } else {
      hipLaunchKernelGGL(k_zero_ghosts<float>, grid, dim3(64), 0, s,
                         static_cast<float *>(grad_u0), mm, desc->g, ld);
    }
    return check_launch("zero ghosts");
  }
  return PSA_OK;
}

}  // namespace

extern "C" {

int psa_adjoint_workspace_bytes(const psa_solver_desc *desc, long long nsteps,
                                int every, size_t *bytes) {
  return psa_adjoint_workspace_bytes_batch(desc, 1, 0, nsteps, every, bytes);
}

int psa_adjoint_workspace_bytes_batch(const psa_solver_desc *desc, long long batch,
                                      long long ld, long long nsteps, int every,
                                      size_t *bytes) {
  int st = check_vjp_desc(desc);
  if (st != PSA_OK) return st;
  st = check_batch(desc, batch, ld);
  if (st != PSA_OK) return st;
  if (bytes == nullptr || nsteps < 0 || every <= 0)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "bad arguments");
  *bytes = adjoint_layout(desc, nsteps, every, batch, ld).bytes;
  return PSA_OK;
}

int psa_ssprk33_forward_checkpointed(const psa_solver_desc *desc,
                                     const void *u0, void *u_final,
                                     long long nsteps, const void *dt,
                                     int every, void *workspace,
                                     size_t workspace_bytes, void *stream) {
  return forward_checkpointed(desc, 1, 0, u0, u_final, nsteps, dt, every, workspace,
                              workspace_bytes, static_cast<hipStream_t>(stream));
}

int psa_ssprk33_forward_checkpointed_batch(const psa_solver_desc *desc, long long batch,
                                           long long ld, const void *u0, void *u_final,
                                           long long nsteps, const void *dt, int every,
                                           void *workspace, size_t workspace_bytes,
                                           void *stream) {
  return forward_checkpointed(desc, batch, ld, u0, u_final, nsteps, dt, every, workspace,
                              workspace_bytes, static_cast<hipStream_t>(stream));
}

int psa_ssprk33_adjoint(const psa_solver_desc *desc, long long nsteps,
                        const void *dt, int every, const void *lam_final,
                        void *grad_u0, void *workspace, size_t workspace_bytes,
                        void *stream) {
  return adjoint(desc, 1, 0, nsteps, dt, every, lam_final, grad_u0, workspace,
                 workspace_bytes, static_cast<hipStream_t>(stream));
}

int psa_ssprk33_adjoint_batch(const psa_solver_desc *desc, long long batch, long long ld,
                              long long nsteps, const void *dt, int every,
                              const void *lam_final, void *grad_u0, void *workspace,
                              size_t workspace_bytes, void *stream) {
  return adjoint(desc, batch, ld, nsteps, dt, every, lam_final, grad_u0, workspace,
                 workspace_bytes, static_cast<hipStream_t>(stream));
}

}  // extern "C"
