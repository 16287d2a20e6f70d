// Host-side rules shared by the launches of the fused forward kernels: tiles,
// which schedule takes a descriptor, and the kernel arguments of a descriptor.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/pyshocks_amd.h"
#include "psa_internal.hpp"
#include "stage_device.hpp"

namespace psa {

inline unsigned int blocks_for(int64_t work, int per_block) {
  return static_cast<unsigned int>((work + per_block - 1) / per_block);
}

struct TileConfig {
  int block;
  int cpt;
  bool pipe;  // stages 1-3: the persistent pipelined kernel
  bool step;  // steps: the whole-step kernel where it applies
};

inline bool aligned16(const void *p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

// Whether the whole-step kernel runs the steps of this descriptor.
inline bool step_applies(const psa_solver_desc *d, TileConfig cfg, int vel) {
  if (!cfg.step || vel == 2 || d->nu != nullptr) return false;
  // the stages of Lax-Friedrichs need the global max|u| of the stage before
  if (d->flux == PSA_FLUX_LAX_FRIEDRICHS) return false;
  if (d->flux == PSA_FLUX_ADVECTION_UPWIND && d->mlp != nullptr) return false;
  if (cfg.block == 256 && cfg.cpt == 1)
    return d->rec == PSA_REC_WENOJS53 && d->flux != PSA_FLUX_ESWENO;
  return cfg.block == 256 && (cfg.cpt == 4 || cfg.cpt == 2);
}

inline TileConfig default_tiles(int dtype) {
  (void)dtype;
  return TileConfig{256, 4, false, true};
}

inline TileConfig tiles_of(const psa_solver_desc *d) {
  TileConfig c = default_tiles(d->dtype);
  // below ~2^20 cells a grid of 1024-cell tiles leaves most of the device
  // idle: half-size tiles double the workgroups in flight
  if (d->n < (int64_t(1) << 20)) c.cpt = 2;
  if (d->block > 0) c.block = d->block;
  if (d->cells_per_thread > 0) c.cpt = d->cells_per_thread;
  if (d->schedule == PSA_SCHEDULE_TILE) c.step = false;
  if (d->schedule == PSA_SCHEDULE_PIPELINE) {
    c.pipe = true;
    c.step = false;
  }
  // below 2^17 cells, one cell per thread where the whole-step kernel takes
  // it (WENO-JS5, learned weights or not): the steps there are latency, and
  // the shorter per-thread chain makes them 8-15% shorter
  if (d->n < (int64_t(1) << 17) && d->block <= 0 && d->cells_per_thread <= 0) {
    TileConfig one = c;
    one.cpt = 1;
    const int vel =
        d->flux != PSA_FLUX_ADVECTION_UPWIND ? 0 : (d->velocity_is_const ? 1 : 2);
    if (step_applies(d, one, vel)) c.cpt = 1;
  }
  return c;
}

template <typename T>
StageArgs<T> make_args(const psa_solver_desc *d) {
  StageArgs<T> a{};
  a.m = d->n + 2 * static_cast<int64_t>(d->g);
  a.n = d->n;
  a.g = d->g;
  a.dx = static_cast<T>(d->dx);
  a.inv_dx = static_cast<T>(1.0) / static_cast<T>(d->dx);
  a.eps = static_cast<T>(d->eps);
  a.vconst = static_cast<T>(d->velocity_const);
  a.vel = static_cast<const T *>(d->velocity);
  if (d->flux == PSA_FLUX_LAX_FRIEDRICHS) {
    a.vel = nullptr;
    a.speed = static_cast<const T *>(d->velocity);
  }
  a.nu = static_cast<const T *>(d->nu);
  a.aligned = 1;
  a.es = d->rec == PSA_REC_ESWENO32 ? 1 : 0;
  a.rec3 = (d->rec == PSA_REC_WENOJS32 || d->rec == PSA_REC_ESWENO32) ? 1 : 0;
  a.muscl = d->rec == PSA_REC_MUSCL ? 1 : 0;
  a.muscls = d->rec == PSA_REC_MUSCLS ? 1 : 0;
  a.es_delta = static_cast<T>(d->es_delta);
  a.nowrap = d->bc == PSA_BC_GIVEN ? 1 : 0;
  a.bcm = (d->bc == PSA_BC_NEUMANN || d->bc == PSA_BC_DIRICHLET) ? d->bc : PSA_BC_PERIODIC;
  a.bc_l = static_cast<T>(d->bc_left);
  a.bc_r = static_cast<T>(d->bc_right);
  a.bc_vals = static_cast<const T *>(d->bc_values);
  a.limiter = d->limiter;
  a.lim_theta = static_cast<T>(d->limiter_theta);
  a.lim_atol = static_cast<T>(d->muscl_atol);
  a.mlp = d->mlp;
  a.tau = static_cast<T>(d->mlp_tau);
  a.sigma = static_cast<T>(d->mlp_sigma);
  return a;
}

inline int vel_mode(const psa_solver_desc *d) {
  if (d->flux != PSA_FLUX_ADVECTION_UPWIND) return 0;
  return d->velocity_is_const ? 1 : 2;
}

// Whether the ring schedule runs the steps of this descriptor (with a
// control block): periodic, at most PSA_RING_MAX_CELLS cells, what the
// whole-step kernel takes without learned weights.
inline bool ring_applies(const psa_solver_desc *d, int vel) {
  if (d->schedule != PSA_SCHEDULE_DEFAULT && d->schedule != PSA_SCHEDULE_RING) return false;
  if (d->bc != PSA_BC_PERIODIC || d->mlp != nullptr || d->nu != nullptr || vel == 2)
    return false;
  if (d->flux == PSA_FLUX_LAX_FRIEDRICHS) return false;
  return d->n >= 8 && d->n <= PSA_RING_MAX_CELLS && d->g >= 2 && d->g <= d->n;
}

// All nsteps steps of a call on the ring schedule (ring_applies), ring.hip.
int launch_ring(const psa_solver_desc *d, const StageArgs<double> &a, long long nsteps,
                hipStream_t stream);
int launch_ring(const psa_solver_desc *d, const StageArgs<float> &a, long long nsteps,
                hipStream_t stream);

// Steps below which its three launches are not worth it (FP64, us a step as
// launches and as a march in calls of four: N = 1500 6.0, 4.2; 16384 6.0, 4.6;
// 374784 8.0, 7.7; 505856 9.0, 9.3, in calls of eight 8.4, 8.1), and the cells that
// a tile's margins need.
constexpr long long kMarchLeastSteps = 4;
constexpr int64_t kMarchLeastCells = 64;

// Whether a call's steps on this descriptor run in one launch that keeps a tile
// per workgroup (march_device.hpp), if the device holds its workgroups at once: the
// default schedule and tiles of a periodic state that the whole-step kernel
// takes, without learned weights, or of the Lax-Friedrichs flux.
inline bool march_applies(const psa_solver_desc *d, TileConfig cfg, int vel) {
  return d->schedule == PSA_SCHEDULE_DEFAULT && d->bc == PSA_BC_PERIODIC && d->block <= 0 &&
         d->cells_per_thread <= 0 && d->mlp == nullptr && d->n >= kMarchLeastCells &&
         (step_applies(d, cfg, vel) ||
          (d->flux == PSA_FLUX_LAX_FRIEDRICHS && d->nu == nullptr));
}

// The steps of a call as a march; k1, k2: scratch arrays of m cells of the
// state's type. PSA_ERR_NOT_IMPLEMENTED (nothing launched) where the state is too
// large for it or the device too small. With a null k2: the same answer, and
// nothing is launched.
int launch_march(const psa_solver_desc *d, const StageArgs<double> &a, long long nsteps,
                 void *k1, void *k2, hipStream_t stream);
int launch_march(const psa_solver_desc *d, const StageArgs<float> &a, long long nsteps,
                 void *k1, void *k2, hipStream_t stream);

// Workgroups the device holds at once for a kernel (CUs x occupancy),
// queried once per kernel and device (the kernel is the template argument,
// so every kernel has a cache of its own).
template <auto Kernel>
unsigned int resident_blocks(int block) {
  constexpr int kMaxDevices = 64;
  static unsigned int cache[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
  if (cache[dev] == 0) {
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, reinterpret_cast<const void *>(Kernel), block, 0) !=
            hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount,
                              dev) != hipSuccess ||
        per_cu <= 0 || cus <= 0) {
      (void)hipGetLastError();
      return 0;
    }
    cache[dev] = static_cast<unsigned int>(per_cu) * static_cast<unsigned int>(cus);
  }
  return cache[dev];
}

}  // namespace psa
