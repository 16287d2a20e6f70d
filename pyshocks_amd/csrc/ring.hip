// The ring schedule: all the steps of a psa_ssprk33_steps call on a small
// periodic state (at most PSA_RING_MAX_CELLS cells) in one launch of one
// workgroup that keeps the state in LDS.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "../../include/pyshocks_amd.h"
#include "psa_internal.hpp"
#include "stage_device.hpp"
#include "step_host.hpp"
#include "wave_device.hpp"

namespace psa {
namespace {

constexpr int kRingMax = PSA_RING_MAX_CELLS;

// Output cells of a wave's window of 64 * CPT cells.
constexpr int ring_out(int cpt) { return 64 * cpt - 2 * kWaveHalo; }

// Up to nsteps steps of the control block's sequence (the decisions of the
// whole-step launches, control_decide_at, from the state's own max|u|); on exit
// u_out holds the state (ghosts filled periodically after a step, or u_in
// as given when no step was taken) and the control block what the
// whole-step schedule leaves (t, m, status, active, dt, umax_bits and the
// final state's max|u| in word 0 of umax_slot). The same bits as the whole-step
// schedule.
//
// Bound by the instructions of one wave (about 300 a step and cell of a thread,
// at 5 to 7 cycles in FP64) and by what the waves wait for each other. A wave
// takes a window of 64 CPT cells through the three stages on its own,
// neighbouring cells a DPP move away, and recomputes the 9 cells on either side
// that its neighbours own; the workgroup meets once a step, to hand over the
// new state and its maximum through LDS. (Cells and states of every thread
// through LDS met six times a step; waves without windows that trade only their
// edges, twice a stage, were slower at every size: a meeting costs as much as
// 20 to 30 instructions.) The maximum and the time step are not needed before
// the stage-1 fluxes are there.
// FP64, Rusanov, us a step before and now: n = 40 1.34, 0.93; 184 1.74, 0.97;
// 256 1.83, 1.34; 440 2.40, 1.32; 512 2.51, 1.72; 1024 4.50, 2.87.
template <typename T, int FLUX, int REC, int CPT>
__global__ __launch_bounds__(1024) void k_ring(StageArgs<T> p, long long nsteps) {
  constexpr int OUT = ring_out(CPT);
  __shared__ T ring[2][kRingMax];
  // the waves' maxima of the new state (entries without a wave stay 0); a NaN
  // in it is told apart, as the maximum passes it by
  __shared__ T s_max[2][16];
  __shared__ int s_nan[2];
  psa_control *ctrl = p.ctrl;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = static_cast<int>(p.n);
  const int g = p.g;

  for (int i = tid; i < n; i += static_cast<int>(blockDim.x)) ring[0][i] = p.uk[g + i];
  if (tid < 32) s_max[tid >> 4][tid & 15] = T(0);
  if (tid < 2) s_nan[tid] = 0;

  // this thread's cells: window cells CPT * lane + r, the window starting 9
  // cells before the wave's output cells
  int cell[CPT];
  bool mine[CPT];
#pragma unroll
  for (int r = 0; r < CPT; ++r) {
    const int k = CPT * lane + r;
    const int i = wave * OUT - kWaveHalo + k;
    mine[r] = k >= kWaveHalo && k < kWaveHalo + OUT && i < n;
    int j = i % n;
    if (j < 0) j += n;
    cell[r] = j;
  }

  const StepParams<T> par(ctrl);
  const bool from_state = ctrl->speed_from_state != 0;
  unsigned long long umax = gather_umax(ctrl);
  double t = ctrl->t;
  long long mstep = ctrl->m;
  int status = ctrl->status;
  bool active = false;
  bool taken = false;
  T dt_last = T(0);
  unsigned long long umax_used = umax;  // max|u| of the last decision
  const MlpSource none{nullptr, nullptr};
  int cur = 0;
  __syncthreads();
  for (long long s = 0; s < nsteps; ++s) {
    T u[CPT], x[CPT], dF[CPT];
#pragma unroll
    for (int r = 0; r < CPT; ++r) u[r] = ring[cur][cell[r]];
    const T top = s_max[cur][lane & 15];
    const int top_nan = s_nan[cur];
    wave_fluxes<T, FLUX, false, REC, CPT>(p, u, dF, none, nullptr);
    if (s > 0 && from_state) umax = top_nan ? nan_bits<T>() : abs_bits(row_max(top));
    T dt = T(0);
    int st;
    umax_used = umax;
    active = control_decide_at<T>(par, t, mstep, status, umax, dt, st);
    status = st;
    // (the same in every lane and wave)
    if (__builtin_amdgcn_readfirstlane(active ? 1 : 0) == 0) break;
    const T lam = stage_lambda<T, FLUX>(p, dt);
#pragma unroll
    for (int r = 0; r < CPT; ++r) x[r] = stage_value<T, 1>(u[r], u[r], lam, dF[r]);
    wave_fluxes<T, FLUX, false, REC, CPT>(p, x, dF, none, nullptr);
#pragma unroll
    for (int r = 0; r < CPT; ++r) x[r] = stage_value<T, 2>(x[r], u[r], lam, dF[r]);
    wave_fluxes<T, FLUX, false, REC, CPT>(p, x, dF, none, nullptr);
    T mx = T(0);
    bool nan = false;
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
      const T v = stage_value<T, 3>(x[r], u[r], lam, dF[r]);
      if (mine[r]) ring[cur ^ 1][cell[r]] = v;
      mx = fmax(mx, mine[r] ? fabs(v) : T(0));
      nan |= mine[r] && isnan(v);
    }
    mx = wave_max(mx);
    if (lane == 63) s_max[cur ^ 1][wave] = mx;
    if (nan) s_nan[cur ^ 1] = 1;
    cur ^= 1;
    t = static_cast<double>(static_cast<T>(t) + dt);
    mstep += 1;
    dt_last = dt;
    taken = true;
    // (the next step writes the buffer this one read, after the barrier)
    __syncthreads();
  }

  if (taken) {
    if (active && from_state)
      umax = s_nan[cur] ? nan_bits<T>() : abs_bits(row_max(s_max[cur][lane & 15]));
    for (int j = tid; j < n + 2 * g; j += static_cast<int>(blockDim.x)) {
      int i = j - g;
      i = i < 0 ? i + n : (i >= n ? i - n : i);
      p.out[j] = ring[cur][i];
    }
  } else {
    for (int j = tid; j < n + 2 * g; j += static_cast<int>(blockDim.x)) p.out[j] = p.uk[j];
  }
  if (tid < 64) {
    if (from_state) ctrl->umax_slot[tid][0] = tid == 0 ? umax : 0ull;
    if (tid == 0) {
      ctrl->t = t;
      ctrl->m = mstep;
      ctrl->status = status;
      ctrl->active = active ? 1 : 0;
      ctrl->umax_bits = umax_used;
      if (taken) ctrl->dt = static_cast<double>(dt_last);
      ctrl->seq_t[0] = t;
      ctrl->seq_m[0] = mstep;
      ctrl->seq_status[0] = status;
    }
  }
}

// Cells per thread: as few as put at most one wave on each SIMD of the CU (a
// second one costs more than another cell per thread: n = 512 2.36 us a step
// with two cells, 1.72 with three), then two.
template <typename T, int FLUX, int REC>
void launch_ring_cells(const StageArgs<T> &a, long long nsteps, hipStream_t s) {
  const int n = static_cast<int>(a.n);
  const auto block = [n](int cpt) {
    return dim3(static_cast<unsigned int>(64 * ((n + ring_out(cpt) - 1) / ring_out(cpt))));
  };
  if (n <= 4 * ring_out(1)) {
    hipLaunchKernelGGL((k_ring<T, FLUX, REC, 1>), dim3(1), block(1), 0, s, a, nsteps);
  } else if (n > 4 * ring_out(2) && n <= 4 * ring_out(3)) {
    hipLaunchKernelGGL((k_ring<T, FLUX, REC, 3>), dim3(1), block(3), 0, s, a, nsteps);
  } else {
    hipLaunchKernelGGL((k_ring<T, FLUX, REC, 2>), dim3(1), block(2), 0, s, a, nsteps);
  }
}

template <typename T, int REC>
int launch_ring_rec(const psa_solver_desc *d, const StageArgs<T> &a, long long nsteps,
                    hipStream_t s) {
  if (d->flux == PSA_FLUX_RUSANOV) {
    launch_ring_cells<T, PSA_FLUX_RUSANOV, REC>(a, nsteps, s);
  } else if (d->flux == PSA_FLUX_BURGERS_UPWIND) {
    launch_ring_cells<T, PSA_FLUX_BURGERS_UPWIND, REC>(a, nsteps, s);
  } else if (d->flux == PSA_FLUX_ENGQUIST_OSHER) {
    launch_ring_cells<T, PSA_FLUX_ENGQUIST_OSHER, REC>(a, nsteps, s);
  } else if (d->flux == PSA_FLUX_ADVECTION_UPWIND) {
    launch_ring_cells<T, PSA_FLUX_ADVECTION_UPWIND, REC>(a, nsteps, s);
  } else if constexpr (REC == 1) {
    if (d->flux != PSA_FLUX_ESWENO)
      return set_error(PSA_ERR_NOT_IMPLEMENTED, "flux not on the ring schedule");
    launch_ring_cells<T, PSA_FLUX_ESWENO, REC>(a, nsteps, s);
  } else {
    return set_error(PSA_ERR_NOT_IMPLEMENTED, "flux not on the ring schedule");
  }
  return check_launch("ring steps");
}

template <typename T>
int launch_ring_t(const psa_solver_desc *d, const StageArgs<T> &a, long long nsteps,
                  hipStream_t s) {
  if (a.rec3) return launch_ring_rec<T, 1>(d, a, nsteps, s);
  if (a.muscl) return launch_ring_rec<T, 2>(d, a, nsteps, s);
  if (a.muscls) return launch_ring_rec<T, 3>(d, a, nsteps, s);
  return launch_ring_rec<T, 0>(d, a, nsteps, s);
}

}  // namespace

int launch_ring(const psa_solver_desc *d, const StageArgs<double> &a, long long nsteps,
                hipStream_t s) {
  return launch_ring_t<double>(d, a, nsteps, s);
}
int launch_ring(const psa_solver_desc *d, const StageArgs<float> &a, long long nsteps,
                hipStream_t s) {
  return launch_ring_t<float>(d, a, nsteps, s);
}

}  // namespace psa
