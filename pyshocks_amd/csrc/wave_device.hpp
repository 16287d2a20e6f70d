// Steps of a tile held by one wave: 64 CPT consecutive cells in registers, CPT
// per lane, the neighbouring cells a DPP move away. No LDS and no barrier
// between the stages; the cells on either side that a step cannot compute
// exactly are recomputed by the neighbouring tiles.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "../../include/pyshocks_amd.h"
#include "stage_device.hpp"

namespace psa {

constexpr int kWaveHalo = 9;  // cells a step takes off either side of a tile

// The value of the lane to the left (lane - 1; 0 in lane 0) or to the right
// (lane + 1; 0 in lane 63): a DPP wave shift.
template <int CTRL>
__device__ __forceinline__ float wave_shift(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double wave_shift(double v) {
  return __hiloint2double(
      __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true),
      __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true));
}
template <typename T>
__device__ __forceinline__ T from_left(T v) {
  return wave_shift<0x138>(v);  // wave_shr:1
}
template <typename T>
__device__ __forceinline__ T from_right(T v) {
  return wave_shift<0x130>(v);  // wave_shl:1
}

// The flux differences of a lane's CPT cells x: the stencils from the
// neighbouring lanes, then reconstruct_any and the face fluxes of step_stage
// (each lane the faces right of its cells, the one to its left from the left
// lane).
template <typename T, int FLUX, bool LEARNED, int REC, int CPT>
__device__ __forceinline__ void wave_fluxes(const StageArgs<T> &p, const T x[CPT], T dF[CPT],
                                            const MlpSource &src, unsigned int *q) {
  constexpr bool ES = FLUX == PSA_FLUX_ESWENO;
  T w[CPT + 4];
  if constexpr (CPT == 1) {
    w[1] = from_left(x[0]);
    w[0] = from_left(w[1]);
    w[3] = from_right(x[0]);
    w[4] = from_right(w[3]);
  } else {
    w[0] = from_left(x[CPT - 2]);
    w[1] = from_left(x[CPT - 1]);
    w[CPT + 2] = from_right(x[0]);
    w[CPT + 3] = from_right(x[1]);
  }
#pragma unroll
  for (int r = 0; r < CPT; ++r) w[2 + r] = x[r];
  T ul[CPT], ur[CPT], om[ES ? CPT : 1];
  reconstruct_any<T, CPT, LEARNED, REC>(p, w, ul, ur, src, q, 0, ES ? om : nullptr);
  const T ulr = from_right(ul[0]);
  T omr = T(0);
  if constexpr (ES) omr = from_right(om[0]);
  T F[CPT + 1];
#pragma unroll
  for (int k = 1; k <= CPT; ++k) {
    const T ulR = k == CPT ? ulr : ul[k < CPT ? k : 0];
    if constexpr (ES) {
      F[k] = flux_burgers_upwind(ur[k - 1], ulR) +
             es_dissipation_w(om[k - 1], k == CPT ? omr : om[k < CPT ? k : 0], w[k + 1],
                              w[k + 2], p.es_delta);
    } else {
      F[k] = stage_flux<T, FLUX>(ur[k - 1], ulR, w[k + 1], w[k + 2], p.vconst);
    }
  }
  F[0] = from_left(F[CPT]);
#pragma unroll
  for (int r = 0; r < CPT; ++r) dF[r] = F[r + 1] - F[r];
}

// Maximum of non-negative values over the wave, in lane 63 (the DPP steps of
// wave_max_u32 on the value itself).
template <int CTRL, int ROWS, typename T>
__device__ __forceinline__ T dpp_max(T v) {
  T o;
  if constexpr (sizeof(T) == 8) {
    o = __hiloint2double(
        __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xF, true),
        __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xF, true));
  } else {
    o = __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xF, true));
  }
  return fmax(v, o);
}
template <typename T>
__device__ __forceinline__ T row_max(T v) {  // of the lane's row of 16, to all of it
  v = dpp_max<0xB1, 0xF>(v);
  v = dpp_max<0x4E, 0xF>(v);
  v = dpp_max<0x124, 0xF>(v);
  return dpp_max<0x128, 0xF>(v);
}
template <typename T>
__device__ __forceinline__ T wave_max(T v) {
  v = row_max(v);
  v = dpp_max<0x142, 0xA>(v);
  return dpp_max<0x143, 0xC>(v);
}

// Output cells of a tile are the cells [LO, 64 CPT - LO), LO a multiple of the
// 16-byte vectors, so that the tiles of an aligned array load and store whole
// vectors.
template <typename T, int CPT>
struct WaveTile {
  static constexpr int C = 64 * CPT;
  static constexpr int LO = sizeof(T) == 8 ? 10 : 12;
  static constexpr int OUT = C - 2 * LO;
  static_assert(LO >= kWaveHalo, "exact output cells");
};

// The lane's first cell in the tile, opaque to the compiler: the masks that come
// from it are made where they are used, not kept in registers over the tiles of
// a loop.
template <int CPT>
__device__ __forceinline__ int wave_cell0() {
  int k0 = CPT * static_cast<int>(threadIdx.x & 63);
  asm volatile("" : "+v"(k0));
  return k0;
}

// Cells base + CPT lane + r of the array u, all of it readable, base a multiple
// of the 16-byte vectors.
template <typename T, int CPT>
__device__ __forceinline__ void wave_load(const T *__restrict__ u, int64_t base, T x[CPT]) {
  constexpr int VN = Vec16<T>::n;
  static_assert(CPT % VN == 0, "whole vectors");
  const T *s = u + base + wave_cell0<CPT>();
#pragma unroll
  for (int r = 0; r < CPT; r += VN) {
    const typename Vec16<T>::type v = load16(s + r);
    x[r] = v.x;
    x[r + 1] = v.y;
    if constexpr (VN == 4) {
      x[r + 2] = v.z;
      x[r + 3] = v.w;
    }
  }
}

// The tile's output cells to u, and the bit pattern of their max|u| (the NaN
// pattern if one is NaN).
template <typename T, int CPT>
__device__ __forceinline__ unsigned long long wave_store(T *__restrict__ u, int64_t base,
                                                         const T x[CPT]) {
  using W = WaveTile<T, CPT>;
  constexpr int VN = Vec16<T>::n;
  const int k0 = wave_cell0<CPT>();
  T *d = u + base + k0;
  T mx = T(0);
  bool nan = false;
#pragma unroll
  for (int r = 0; r < CPT; r += VN) {
    typename Vec16<T>::type v;
    if constexpr (VN == 2) {
      v = {x[r], x[r + 1]};
    } else {
      v = {x[r], x[r + 1], x[r + 2], x[r + 3]};
    }
    const bool out = k0 + r >= W::LO && k0 + r < W::C - W::LO;
    if (out) store16(d + r, v);
#pragma unroll
    for (int k = r; k < r + VN; ++k) {
      mx = fmax(mx, out ? fabs(x[k]) : T(0));
      nan |= out && isnan(x[k]);
    }
  }
  return nan ? nan_bits<T>() : abs_bits(mx);
}

// One SSP-RK3 step (timestepping.py:312-320) of the tile: u is u^n on entry and
// u^(n+1) on return, exact on all but the 9 outermost cells of either side, the
// bits of the stage kernels.
template <typename T, int FLUX, bool LEARNED, int REC, int CPT>
__device__ __forceinline__ void wave_step(const StageArgs<T> &p, T u[CPT], T dt,
                                          const MlpSource &src, unsigned int *q) {
  const T lam = stage_lambda<T, FLUX>(p, dt);
  T x[CPT];
#pragma unroll
  for (int r = 0; r < CPT; ++r) x[r] = u[r];
  // (one copy of the stage's code: it fills a good part of the instruction
  // cache)
#pragma unroll 1
  for (int stage = 1; stage <= 3; ++stage) {
    T dF[CPT];
    wave_fluxes<T, FLUX, LEARNED, REC, CPT>(p, x, dF, src, q);
    if (stage == 1) {
#pragma unroll
      for (int r = 0; r < CPT; ++r) x[r] = stage_value<T, 1>(x[r], u[r], lam, dF[r]);
    } else if (stage == 2) {
#pragma unroll
      for (int r = 0; r < CPT; ++r) x[r] = stage_value<T, 2>(x[r], u[r], lam, dF[r]);
    } else {
#pragma unroll
      for (int r = 0; r < CPT; ++r) x[r] = stage_value<T, 3>(x[r], u[r], lam, dF[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < CPT; ++r) u[r] = x[r];
}

}  // namespace psa
