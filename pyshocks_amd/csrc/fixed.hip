// Fixed-dt SSP-RK3 steps (timestepping.py:312-320) of the adjoint's forward and
// recompute passes: several steps of a tile per launch, without step control.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "../../include/pyshocks_amd.h"
#include "psa_internal.hpp"
#include "stage_device.hpp"
#include "step_host.hpp"

namespace psa {
namespace {

constexpr int kBlock = 256;
// (a tile of 256 cells then has 56 output cells left)
constexpr int kMostSteps = 12;

template <typename T>
struct FixedArgs {
  const T *in;          // the state before the first step
  T *out;               // the state after step s at out + s * stride (stride
  T *k1;                //   0: after the last one only), its stage states at
  T *k2;                //   k1, k2 + s * stride, or null
  const T *dt;          // instance b: dt[b]
  int64_t stride;
  int64_t bstride;      // instance b = blockIdx.y: at b * bstride of every array
  int nsub;             // steps of this launch
  int lo, to;           // a tile's output cells [lo, lo + to) of its C + 8
  int aligned;          // every array and stride 16-byte aligned
};

// nsub steps of the tile of blockIdx.x: the workgroup holds C + 8 cells of the
// state (step_tile_ctl's layout) and computes C of them in every stage; each step
// takes 9 exact cells off either side (step_tile_ctl), so after nsub of them
// the cells [11 + 9 (nsub - 1), C - 3 - 9 (nsub - 1)) are exact and the output
// cells lie inside. The neighbouring tiles recompute the margins; the results
// are the whole-step kernel's bit for bit, whatever nsub.
//
// One step per launch is all launch, load and drain at the sizes of a single
// gradient (N = 16384: 4.0 us a step, of which the three stages are 1.6 us),
// on a device that is nearly idle, so the recomputation is free there and
// several steps share that cost.
// MANY: more than one step.
template <typename T, int FLUX, int VEL, int CPT, bool LEARNED, bool MANY>
__global__ __attribute__((amdgpu_flat_work_group_size(1, kBlock),
                          amdgpu_waves_per_eu((step_min_waves<T, LEARNED, 0>()))))
void k_fixed_steps(StageArgs<T> p, FixedArgs<T> f) {
  using SM = StepSmem<T, kBlock, CPT>;
  constexpr int C = SM::C;
  constexpr int L = SM::L;
  __shared__ SM sm;
  __shared__ unsigned int q[LEARNED ? (kBlock / 64) * learned_queue_words<CPT>() : 1];
  const int tid = threadIdx.x;
  const int g = p.g;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * f.to - f.lo;
  const int64_t off = static_cast<int64_t>(blockIdx.y) * f.bstride;
  const T *in = f.in + off;
  const T dt = f.dt[blockIdx.y];

  const bool fast = f.aligned != 0 && base >= g && base + L <= p.m - g;
  if (fast) {
    Chunks<T, kBlock, L / Vec16<T>::n> cu;
    cu.load(in + base, tid);
    cu.store(sm.x0, tid);
  } else {
    const PeriodicSpan span(base, p.n, g);
    for (int j = tid; j < L; j += kBlock) sm.x0[j] = span.load(in, j);
  }
  // entries without a neighbouring thread (outside the exact ranges)
  if (tid < 8) sm.x1[tid < 4 ? tid : C + tid] = T(0);
  if (tid == 0) {
    sm.urL[0] = T(0);
    sm.ulF[kBlock] = T(0);
  }
  __syncthreads();

  const int j0 = 4 + CPT * tid;
  const int hi = f.lo + f.to;
  T un[CPT], val[CPT];
#pragma unroll
  for (int r = 0; r < CPT; ++r) un[r] = sm.x0[j0 + r];
  const MlpSource src{p.mlp, nullptr};
  unsigned long long unused = 0;
  for (int s = 0; MANY ? s < f.nsub : s < 1; ++s) {
    const int64_t at = off + s * f.stride;
    step_stage<T, FLUX, VEL, kBlock, CPT, 1, LEARNED>(p, sm.x0, sm, dt, un, val, src, q);
#pragma unroll
    for (int r = 0; r < CPT; ++r) sm.x1[j0 + r] = val[r];
    if (f.k1 != nullptr)
      step_store<T, kBlock, CPT, false>(p, base, fast, val, f.k1 + at, unused, f.lo, hi);
    __syncthreads();
    step_stage<T, FLUX, VEL, kBlock, CPT, 2, LEARNED>(p, sm.x1, sm, dt, un, val, src, q);
#pragma unroll
    for (int r = 0; r < CPT; ++r) sm.x0[j0 + r] = val[r];
    if (f.k2 != nullptr)
      step_store<T, kBlock, CPT, false>(p, base, fast, val, f.k2 + at, unused, f.lo, hi);
    __syncthreads();
    step_stage<T, FLUX, VEL, kBlock, CPT, 3, LEARNED>(p, sm.x0, sm, dt, un, val, src, q);
    if (!MANY || f.stride != 0 || s == f.nsub - 1)
      step_store<T, kBlock, CPT, false>(p, base, fast, val, f.out + at, unused, f.lo, hi);
    if constexpr (MANY) {
      // (every read of x0 ended before the exchange barrier of stage 3)
#pragma unroll
      for (int r = 0; r < CPT; ++r) {
        sm.x0[j0 + r] = val[r];
        un[r] = val[r];
      }
      __syncthreads();
    }
  }
}

// First output cell of a tile and output cells of a tile for nsub steps
// (multiples of 4, so that a fast tile stays 16-byte aligned).
constexpr int fixed_lo(int nsub) { return (11 + 9 * (nsub - 1) + 3) / 4 * 4; }
constexpr int fixed_to(int c, int nsub) {
  return (c - 3 - 9 * (nsub - 1) - fixed_lo(nsub)) / 4 * 4;
}

template <typename T, int FLUX, int VEL, int CPT, bool LEARNED>
int launch_fixed(const StageArgs<T> &p, FixedArgs<T> f, long long batch, hipStream_t s) {
  constexpr int C = kBlock * CPT;
  f.lo = fixed_lo(f.nsub);
  f.to = fixed_to(C, f.nsub);
  const dim3 grid(blocks_for(p.m, f.to), static_cast<unsigned int>(batch));
  if constexpr (CPT <= 2) {
    if (f.nsub > 1) {
      hipLaunchKernelGGL((k_fixed_steps<T, FLUX, VEL, CPT, LEARNED, true>), grid, dim3(kBlock),
                         0, s, p, f);
      return check_launch("fixed steps");
    }
  }
  hipLaunchKernelGGL((k_fixed_steps<T, FLUX, VEL, CPT, LEARNED, false>), grid, dim3(kBlock), 0,
                     s, p, f);
  return check_launch("fixed steps");
}

template <typename T, int FLUX, int VEL, bool LEARNED>
int launch_fixed_tiles(const StageArgs<T> &p, const FixedArgs<T> &f, int cpt, long long batch,
                       hipStream_t s) {
  if (cpt == 4) return launch_fixed<T, FLUX, VEL, 4, LEARNED>(p, f, batch, s);
  if (cpt == 2) return launch_fixed<T, FLUX, VEL, 2, LEARNED>(p, f, batch, s);
  return launch_fixed<T, FLUX, VEL, 1, LEARNED>(p, f, batch, s);
}

// The tiles of the fixed steps of a batch: those of the descriptor; a batch
// fills the device with its instances, so there the one-cell tiles of the
// small single grids give way to two cells per thread (the learned step 6%
// faster in batches of 64, the plain one the same).
TileConfig fixed_tiles(const psa_solver_desc *d, long long batch) {
  TileConfig cfg = tiles_of(d);
  if (batch > 1 && cfg.cpt == 1 && d->cells_per_thread <= 0) cfg.cpt = 2;
  return cfg;
}

template <typename T>
int launch_fixed_desc(const psa_solver_desc *d, const void *u_in, void *u_out, void *k1,
                      void *k2, long long nsub, int64_t stride, const void *dt,
                      hipStream_t s, long long batch, int64_t ld, int cpt) {
  const StageArgs<T> p = make_args<T>(d);
  FixedArgs<T> f{};
  f.in = static_cast<const T *>(u_in);
  f.out = static_cast<T *>(u_out);
  f.k1 = static_cast<T *>(k1);
  f.k2 = static_cast<T *>(k2);
  f.dt = static_cast<const T *>(dt);
  f.stride = stride;
  f.bstride = ld;
  f.nsub = static_cast<int>(nsub);
  f.aligned = aligned16(u_in) && aligned16(u_out) && aligned16(k1) && aligned16(k2) &&
              (ld | stride) * static_cast<int64_t>(sizeof(T)) % 16 == 0;
  if (d->mlp != nullptr) {
    if (d->flux == PSA_FLUX_RUSANOV)
      return launch_fixed_tiles<T, PSA_FLUX_RUSANOV, 0, true>(p, f, cpt, batch, s);
    if (d->flux == PSA_FLUX_ENGQUIST_OSHER)
      return launch_fixed_tiles<T, PSA_FLUX_ENGQUIST_OSHER, 0, true>(p, f, cpt, batch, s);
    return launch_fixed_tiles<T, PSA_FLUX_BURGERS_UPWIND, 0, true>(p, f, cpt, batch, s);
  }
  if (d->flux == PSA_FLUX_RUSANOV)
    return launch_fixed_tiles<T, PSA_FLUX_RUSANOV, 0, false>(p, f, cpt, batch, s);
  if (d->flux == PSA_FLUX_BURGERS_UPWIND)
    return launch_fixed_tiles<T, PSA_FLUX_BURGERS_UPWIND, 0, false>(p, f, cpt, batch, s);
  if (d->flux == PSA_FLUX_ENGQUIST_OSHER)
    return launch_fixed_tiles<T, PSA_FLUX_ENGQUIST_OSHER, 0, false>(p, f, cpt, batch, s);
  return launch_fixed_tiles<T, PSA_FLUX_ADVECTION_UPWIND, 1, false>(p, f, cpt, batch, s);
}

}  // namespace

// Measured (FP64, Rusanov; us a step with 1 step per launch and with the chosen
// number): one instance of 256 cells 3.67 -> 1.71, of 16384 3.95 -> 1.85, of
// 65536 4.19 -> 2.52; 16 instances of 16384 6.85 -> 4.45 (two cells per thread).
int fixed_steps_per_launch(const psa_solver_desc *d, long long batch) {
  const TileConfig cfg = fixed_tiles(d, batch);
  if (!step_applies(d, cfg, vel_mode(d))) return 0;
  // (the tiles of four cells per thread are for grids that fill the device)
  if (cfg.cpt > 2) return 1;
  const int64_t m = d->n + 2 * static_cast<int64_t>(d->g);
  const StepCost cost = cfg.cpt == 1 ? StepCost{2.4, 1.15, 0.45} : StepCost{2.9, 1.6, 0.8};
  return best_steps(cost, kMostSteps, [&](int k) {
    return static_cast<long long>(blocks_for(m, fixed_to(kBlock * cfg.cpt, k))) * batch;
  });
}

int steps_fixed_dt(const psa_solver_desc *d, const void *u_in, void *u_out, void *k1,
                   void *k2, long long nsub, int64_t stride, const void *dt,
                   hipStream_t stream, long long batch, int64_t ld) {
  const TileConfig cfg = fixed_tiles(d, batch);
  if (!step_applies(d, cfg, vel_mode(d))) return PSA_ERR_NOT_IMPLEMENTED;
  if (batch < 1 || batch > 65535)
    return set_error(PSA_ERR_INVALID_ARGUMENT, "batch must be in [1, 65535]");
  if (nsub < 1 || nsub > kMostSteps || (nsub > 1 && cfg.cpt > 2))
    return set_error(PSA_ERR_INVALID_ARGUMENT, "too many steps in a launch");
  if (d->dtype == PSA_FLOAT64)
    return launch_fixed_desc<double>(d, u_in, u_out, k1, k2, nsub, stride, dt, stream, batch,
                                     ld, cfg.cpt);
  return launch_fixed_desc<float>(d, u_in, u_out, k1, k2, nsub, stride, dt, stream, batch,
                                  ld, cfg.cpt);
}

}  // namespace psa
