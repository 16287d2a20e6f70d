// The march schedule: all the steps of a psa_ssprk33_steps call on a mid-size
// periodic state in one launch, the state in the registers of its waves
// throughout (march.hip in FP64, march_f32.hip in FP32).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "../../include/pyshocks_amd.h"
#include "exchange_device.hpp"
#include "psa_internal.hpp"
#include "stage_device.hpp"
#include "step_host.hpp"
#include "wave_device.hpp"

namespace psa {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kHalo = kWaveHalo;
constexpr int kMarchMaxTiles = 256;
constexpr double kMarchWaitSeconds = 600.0;

// Before the steps: words that no step waits for.
__global__ void k_march_init(unsigned long long *words, int nmax, int nall, int *abort) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < nall) words[i] = i < nmax ? kTurn : 0ull;
  if (i == 0) *abort = 0;
}

template <typename T>
struct MarchArgs {
  const T *in;
  T *out;
  Exchange<T> x;
  int *abort;
  long long nsteps;
  long long wait_ticks;  // limit of a wait, in wall-clock ticks
};

// Whether a wait that began then may go on (asked every kSpins loads: the flag's
// load would double the time between two looks at the words).
constexpr unsigned int kSpins = 256;

template <typename T>
__device__ __forceinline__ bool waits(const MarchArgs<T> &f, long long began) {
  return wall_clock64() - began < f.wait_ticks &&
         __hip_atomic_load(f.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
}

// Up to nsteps steps of the control block's sequence with the decisions of the
// whole-step launches (control_decide_at); the state, the control block and
// every value in between are the whole-step schedule's (Lax-Friedrichs: the
// stage schedule's) bit for bit. Wave w of all the launch's waves holds the cells
// [w n / waves, (w + 1) n / waves) and 9 on either side in registers (wave
// tiles); after a step a workgroup publishes its new maximum and edge cells,
// waits for every tile's maximum and its neighbours' edges, and its waves hand
// each other theirs through LDS. Lax-Friedrichs takes the maximum of every
// stage's output the same way, the speed of the next stage's flux.
//
// Every workgroup has to be resident for the waits to end: the launch takes no
// more than a quarter of what the device holds (launch_march_cells), so that the
// marches of four streams fit together, kernels that end by themselves only delay
// it, and a wait of ten minutes gives up for all (status PSA_ERR_HIP).
//
// Bound by latency up to some 10^5 cells: the instructions of one wave, as in
// the ring schedule, and one exchange through memory (1.1 to 1.7 us), against a
// launch, load, control block and drain per step; above, by the FP64 rate of the
// few waves. FP64, Rusanov, WENO-JS5, us a step as a launch each and as a march:
// N = 1500 5.23, 2.58; 16384 5.05, 2.90; 47104 5.14, 3.30; 112640 5.47, 3.82;
// 243712 6.50, 4.81; 374784 7.46, 6.11; 505856 8.41, 7.18 (FP32 4.79, 2.44 to 6.55,
// 6.09). Lax-Friedrichs, as three launches a step and as a march: N = 184 12.9,
// 2.5; 16384 15.3, 6.5; 112640 15.7, 8.4; 505856 19.8, 12.3 (FP32 12.6, 2.3 to
// 17.5, 10.6). With learned weights the network's latency rules and both take the
// same, so they stay on the step kernel.
template <typename T, int FLUX, int REC, int CPT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_march(
    StageArgs<T> p, MarchArgs<T> f) {
  using X = Exchange<T>;
  constexpr bool LF = FLUX == PSA_FLUX_LAX_FRIEDRICHS;
  // slot w + 1: the first and the last 9 cells of wave w, slots 0 and kWaves +
  // 1: the left tile's last ones and the right tile's first ones
  // (two sets, used in turn: a wave may be a step ahead of another's reads)
  __shared__ T s_edges[2][kWaves + 2][2][kHalo];
  // u^n of a lane's cells where the registers do not hold both
  constexpr bool ULDS = sizeof(T) == 8 && CPT > 4;
  __shared__ T s_u[ULDS ? CPT : 1][ULDS ? kBlock : 1];
  __shared__ unsigned long long s_red[kWaves], s_top[kWaves];
  __shared__ int s_abort;
  __shared__ __align__(16) unsigned char s_params[sizeof(StepParams<T>)];
  psa_control *ctrl = p.ctrl;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = p.g;
  const int tiles = f.x.tiles;
  const int tile = static_cast<int>(blockIdx.x);
  const int64_t gw = static_cast<int64_t>(tile) * kWaves + wave;
  const int64_t start = p.n * gw / (tiles * kWaves);
  const int cnt = static_cast<int>(p.n * (gw + 1) / (tiles * kWaves) - start);
  const int left = tile == 0 ? tiles - 1 : tile - 1;
  const int right = tile == tiles - 1 ? 0 : tile + 1;
  // the slots that hold the cells left and right of this wave's
  const int lslot = tiles == 1 && wave == 0 ? kWaves : wave;
  const int rslot = tiles == 1 && wave == kWaves - 1 ? 1 : wave + 2;
  int k0 = CPT * lane;  // window cell of x[0]; own cells are [9, 9 + cnt)

  T x[CPT];
  {
    const PeriodicSpan span(start + g - kHalo, p.n, g);
#pragma unroll
    for (int r = 0; r < CPT; ++r) x[r] = span.load(f.in, k0 + r);
  }
  if (tid == 0) s_abort = 0;
  // (in LDS: read once a step, the registers are for the cells)
  StepParams<T> &par = *reinterpret_cast<StepParams<T> *>(s_params);
  if (tid == 0) par = StepParams<T>(ctrl);
  const bool from_state = ctrl->speed_from_state != 0;
  unsigned long long umax = gather_umax(ctrl);
  unsigned long long umax_used = umax;  // max|u| of the last decision
  double t = ctrl->t;
  long long mstep = ctrl->m;
  int status = ctrl->status;
  bool active = false;
  bool taken = false;
  T dt_last = T(0);
  unsigned int turns = 0;  // exchanges so far
  StageArgs<T> pl = p;
  const MlpSource none{nullptr, nullptr};
  __syncthreads();

  // The maximum of |x| over the own cells of all waves; with s_edge, also the
  // neighbour tiles' edge cells of the step of the tag into its outer slots. False: the
  // wait was given up. Every thread of the launch takes part.
  auto exchange = [&](unsigned long long tag, T (*s_edge)[2][kHalo],
                      unsigned long long &top) -> bool {
    const int set = static_cast<int>(turns & 1u);
    const unsigned long long turn = (turns & 2u) != 0 ? kTurn : 0ull;
    ++turns;
    T mx = T(0);
    bool nan = false;
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
      const int o = k0 + r - kHalo;
      const bool mine = o >= 0 && o < cnt;
      mx = fmax(mx, mine ? fabs(x[r]) : T(0));
      nan |= mine && isnan(x[r]);
    }
    mx = wave_max(mx);
    const bool any_nan = __any(nan);
    if (lane == 63) s_red[wave] = any_nan ? nan_bits<T>() : abs_bits(mx);
    __syncthreads();
    unsigned long long v = s_red[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) v = s_red[w] > v ? s_red[w] : v;
    if (tiles == 1) {
      top = v;
      // (s_red is written again after the next stage's or step's first barrier
      // only if every thread has read it)
      __syncthreads();
      return true;
    }
    if (tid == 0) put(f.x.max_word(set, tile), turn | v);

    // wait for the neighbours' edges (the last wave) and every maximum (64
    // tiles a wave)
    const long long began = wall_clock64();
    bool ok = true;
    if (s_edge != nullptr && wave == kWaves - 1) {
      const bool mine = lane < 2 * X::SIDE;
      const int side = lane < X::SIDE ? 0 : 1;
      const int k = lane - side * X::SIDE;
      // the cells left of the tile are the left tile's last ones
      const unsigned long long *w =
          mine ? f.x.cells(set, side == 0 ? left : right, side == 0 ? 1 : 0) + k : nullptr;
      unsigned long long c = tag;
      for (unsigned int spin = 1;; ++spin) {
        if (mine) c = get(w);
        const bool there = (c & 0xFFFFFFFF00000000ull) == tag;
        if (__all(there)) break;
        if (spin % kSpins == 0 && !(ok = waits(f, began))) break;
      }
      const unsigned int bits = static_cast<unsigned int>(c);
      T *to = side == 0 ? s_edge[0][1] : s_edge[kWaves + 1][0];
      if constexpr (X::NW == 2) {
        const unsigned int hi = __shfl_down(bits, 1, 64);
        if (mine && (k & 1) == 0)
          to[k >> 1] = __hiloint2double(static_cast<int>(hi), static_cast<int>(bits));
      } else {
        if (mine) to[k] = __uint_as_float(bits);
      }
    }
    unsigned long long most = 0;
    if (64 * wave < tiles) {
      const bool mine = 64 * wave + lane < tiles;
      const unsigned long long *w = f.x.max_word(set, mine ? 64 * wave + lane : 0);
      unsigned long long c = turn;
      for (unsigned int spin = 1; ok; ++spin) {
        if (mine) c = get(w);
        if (__all((c & kTurn) == turn)) break;
        if (spin % kSpins == 0) ok = waits(f, began);
      }
      most = wave_max_u64(c & ~kTurn);
    }
    if (lane == 0) {
      s_top[wave] = most;
      if (!ok) s_abort = 1;
    }
    __syncthreads();
    top = s_top[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) top = s_top[w] > top ? s_top[w] : top;
    if (s_abort == 0) return true;
    // a workgroup is not running: everyone leaves
    if (tid == 0) __hip_atomic_store(f.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return false;
  };

  for (long long s = 0; s < f.nsteps; ++s) {
    // (k0 opaque: the addresses of the exchange made anew each step instead of
    // kept in registers over all of them)
    asm volatile("" : "+v"(k0));
    T u[ULDS ? 1 : CPT];
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
      if constexpr (ULDS) s_u[r][tid] = x[r];
      else u[r] = x[r];
    }
    const auto u_of = [&](int r) -> T {
      if constexpr (ULDS) return s_u[r][tid];
      else return u[r];
    };
    T dt = T(0), lam = T(0);
    bool ok = true;
    T (*s_edge)[2][kHalo] = s_edges[s & 1];
    // (one copy of the stage's code where the work, not the latency, counts)
    constexpr int COPIES = CPT <= 2 ? 3 : 1;
#pragma unroll COPIES
    for (int stage = 1; stage <= 3; ++stage) {
      T dF[CPT];
      if constexpr (LF) {
        if (stage == 1) pl.vconst = from_bits<T>(umax);
      }
      wave_fluxes<T, FLUX, false, REC, CPT>(pl, x, dF, none, nullptr);
      if (stage == 1) {
        int st;
        umax_used = umax;
        active = control_decide_at<T>(par, t, mstep, status, umax, dt, st);
        status = st;
        // (the same in every lane, wave and workgroup)
        if (__builtin_amdgcn_readfirstlane(active ? 1 : 0) == 0) break;
        lam = stage_lambda<T, FLUX>(pl, dt);
#pragma unroll
        for (int r = 0; r < CPT; ++r) x[r] = stage_value<T, 1>(x[r], x[r], lam, dF[r]);
      } else if (stage == 2) {
#pragma unroll
        for (int r = 0; r < CPT; ++r) x[r] = stage_value<T, 2>(x[r], u_of(r), lam, dF[r]);
      } else {
#pragma unroll
        for (int r = 0; r < CPT; ++r) x[r] = stage_value<T, 3>(x[r], u_of(r), lam, dF[r]);
      }
      if constexpr (LF) {
        if (stage < 3) {
          unsigned long long top;
          ok = exchange(0ull, nullptr, top);
          if (!ok) break;
          pl.vconst = from_bits<T>(top);
        }
      }
    }
    if (__builtin_amdgcn_readfirstlane(active ? 1 : 0) == 0) break;
    if (ok) {
      t = static_cast<double>(static_cast<T>(t) + dt);
      mstep += 1;
      dt_last = dt;
      taken = true;

      // ---- publish the edges (LDS for the tile's waves, words for its
      // neighbours), then trade the maximum
      const unsigned long long tag = static_cast<unsigned long long>(
                                         static_cast<unsigned int>(s + 1))
                                     << 32;
      const int set = static_cast<int>(turns & 1u);
#pragma unroll
      for (int r = 0; r < CPT; ++r) {
        const int o = k0 + r - kHalo;  // own cell
        if (o >= 0 && o < kHalo) {
          s_edge[wave + 1][0][o] = x[r];
          if (wave == 0 && tiles > 1) {
#pragma unroll
            for (int k = 0; k < X::NW; ++k)
              put(f.x.cells(set, tile, 0) + X::NW * o + k, tag | word_of(x[r], k));
          }
        }
        if (o >= cnt - kHalo && o < cnt) {
          const int e = o - (cnt - kHalo);
          s_edge[wave + 1][1][e] = x[r];
          if (wave == kWaves - 1 && tiles > 1) {
#pragma unroll
            for (int k = 0; k < X::NW; ++k)
              put(f.x.cells(set, tile, 1) + X::NW * e + k, tag | word_of(x[r], k));
          }
        }
      }
      unsigned long long top;
      ok = exchange(tag, s_edge, top);
      if (from_state) umax = top;
    }
    if (!ok) {
      status = PSA_ERR_HIP;
      break;
    }
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
      const int k = k0 + r;
      if (k < kHalo) x[r] = s_edge[lslot][1][k];
      if (k >= kHalo + cnt && k < 2 * kHalo + cnt) x[r] = s_edge[rslot][0][k - kHalo - cnt];
    }
  }

  // ---- the wave's cells and their ghost images
  if (taken || f.out != f.in) {
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
      const int o = k0 + r - kHalo;
      if (o < 0 || o >= cnt) continue;
      const int64_t i = start + o;
      f.out[g + i] = x[r];
      if (taken) {
        if (i < g) f.out[g + p.n + i] = x[r];
        if (i >= p.n - g) f.out[g + i - p.n] = x[r];
      }
    }
    if (!taken && tile == 0) {
      // no step: the ghost cells as given
      for (int k = tid; k < 2 * g; k += kBlock) {
        const int64_t c = k < g ? k : p.n + k;
        f.out[c] = f.in[c];
      }
    }
  }
  if (tile == 0 && tid < 64) {
    // (without a step, tiles that start later still read the slots: a mixture of
    // old and new ones could have them take a step that the others do not)
    if (from_state && taken) ctrl->umax_slot[tid][0] = tid == 0 ? umax : 0ull;
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

// Cells of a workgroup with CPT cells per lane.
constexpr int march_cells(int cpt) { return kWaves * (64 * cpt - 2 * kHalo); }

template <typename T, int FLUX, int REC, int CPT>
int launch_march_cells(const StageArgs<T> &a, MarchArgs<T> f, void *scratch, hipStream_t s) {
  const int tiles =
      static_cast<int>((a.n + march_cells(CPT) - 1) / march_cells(CPT));
  const unsigned int resident = resident_blocks<k_march<T, FLUX, REC, CPT>>(kBlock);
  if (resident < 4u * static_cast<unsigned int>(tiles)) return PSA_ERR_NOT_IMPLEMENTED;
  // the exchange words and the abort flag in the caller's scratch array
  // (no scratch: the caller asks whether it would run)
  const uintptr_t at =
      (reinterpret_cast<uintptr_t>(scratch) + 127u) & ~static_cast<uintptr_t>(127);
  const int count = tiles > 1 ? Exchange<T>::count(tiles) : 0;
  const size_t need = sizeof(unsigned long long) * static_cast<size_t>(count) + sizeof(int) +
                      (at - reinterpret_cast<uintptr_t>(scratch));
  if (need > static_cast<size_t>(a.m) * sizeof(T)) return PSA_ERR_NOT_IMPLEMENTED;
  if (scratch == nullptr) return PSA_OK;
  f.x.words = reinterpret_cast<unsigned long long *>(at);
  f.x.tiles = tiles;
  f.abort = reinterpret_cast<int *>(f.x.words + count);
  if (tiles > 1) {
    hipLaunchKernelGGL(k_march_init, dim3(blocks_for(count, 256)), dim3(256), 0, s, f.x.words,
                       2 * tiles * Exchange<T>::SPREAD, count, f.abort);
    const int st = check_launch("march init");
    if (st != PSA_OK) return st;
  }
  hipLaunchKernelGGL((k_march<T, FLUX, REC, CPT>), dim3(static_cast<unsigned int>(tiles)),
                     dim3(kBlock), 0, s, a, f);
  return check_launch("march steps");
}

// The fewest cells per lane that leave the launch within kMarchMaxTiles
// workgroups: a wave's instructions cost more than tiles to exchange with (FP64,
// N = 16384, 1 to 8 cells per lane: 2.90, 3.35, 4.20, 5.29, 6.37 us a step). With
// Lax-Friedrichs' three exchanges a step one tile alone wins as long as it takes
// no more than 4 cells per lane (N = 952: 4.2 us against 5.7 with 6 tiles; of
// 1500 cells 6.5 against 5.6). The line to the whole-step launches lies where
// they are as fast: MUSCL, with more temporaries per cell, 243712 cells (6.55
// against 7.09; with 6 cells per lane 8.5), else 505856 (7.2 against 8.4, FP32 6.1
// against 6.5; FP32 with 16 cells per lane 8.9); the stage launches of
// Lax-Friedrichs take longer up to the largest tiles (FP32, N = 1030144: 14.3
// against 21.5; FP64, N = 505856: 12.3 against 19.8).
template <typename T, int FLUX, int REC>
int launch_march_tiles(const StageArgs<T> &a, const MarchArgs<T> &f, void *scratch,
                       hipStream_t s) {
  constexpr bool LF = FLUX == PSA_FLUX_LAX_FRIEDRICHS;
  constexpr int MOST = LF ? (sizeof(T) == 4 ? 16 : 8) : (REC >= 2 ? 4 : 8);
  const int most = LF && a.n <= march_cells(4) ? 1 : kMarchMaxTiles;
  const auto fits = [&](int cpt) {
    return a.n <= static_cast<int64_t>(most) * march_cells(cpt);
  };
  if (fits(1)) return launch_march_cells<T, FLUX, REC, 1>(a, f, scratch, s);
  if (fits(2)) return launch_march_cells<T, FLUX, REC, 2>(a, f, scratch, s);
  if (fits(4)) return launch_march_cells<T, FLUX, REC, 4>(a, f, scratch, s);
  if constexpr (MOST >= 8) {
    if (fits(6)) return launch_march_cells<T, FLUX, REC, 6>(a, f, scratch, s);
    if (fits(8)) return launch_march_cells<T, FLUX, REC, 8>(a, f, scratch, s);
  }
  if constexpr (MOST >= 16) {
    if (fits(16)) return launch_march_cells<T, FLUX, REC, 16>(a, f, scratch, s);
  }
  return PSA_ERR_NOT_IMPLEMENTED;
}

template <typename T, int REC>
int launch_march_rec(const psa_solver_desc *d, const StageArgs<T> &a, const MarchArgs<T> &f,
                     void *scratch, hipStream_t s) {
  if (d->flux == PSA_FLUX_RUSANOV)
    return launch_march_tiles<T, PSA_FLUX_RUSANOV, REC>(a, f, scratch, s);
  if (d->flux == PSA_FLUX_BURGERS_UPWIND)
    return launch_march_tiles<T, PSA_FLUX_BURGERS_UPWIND, REC>(a, f, scratch, s);
  if (d->flux == PSA_FLUX_ENGQUIST_OSHER)
    return launch_march_tiles<T, PSA_FLUX_ENGQUIST_OSHER, REC>(a, f, scratch, s);
  if (d->flux == PSA_FLUX_LAX_FRIEDRICHS)
    return launch_march_tiles<T, PSA_FLUX_LAX_FRIEDRICHS, REC>(a, f, scratch, s);
  if constexpr (REC == 1) {
    if (d->flux == PSA_FLUX_ESWENO)
      return launch_march_tiles<T, PSA_FLUX_ESWENO, REC>(a, f, scratch, s);
  }
  return launch_march_tiles<T, PSA_FLUX_ADVECTION_UPWIND, REC>(a, f, scratch, s);
}

template <typename T>
int launch_march_t(const psa_solver_desc *d, const StageArgs<T> &a, long long nsteps,
                   void *scratch, hipStream_t s) {
  MarchArgs<T> f{};
  f.in = a.uk;
  f.out = a.out;
  f.nsteps = nsteps;
  int dev = 0, rate_khz = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess ||
      rate_khz <= 0) {
    (void)hipGetLastError();
    rate_khz = 100000;  // 100 MHz
  }
  f.wait_ticks = static_cast<long long>(kMarchWaitSeconds * 1000.0 * rate_khz);
  if (a.rec3) return launch_march_rec<T, 1>(d, a, f, scratch, s);
  if (a.muscl) return launch_march_rec<T, 2>(d, a, f, scratch, s);
  if (a.muscls) return launch_march_rec<T, 3>(d, a, f, scratch, s);
  return launch_march_rec<T, 0>(d, a, f, scratch, s);
}

}  // namespace
}  // namespace psa
