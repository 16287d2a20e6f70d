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
constexpr double kMarchGateSeconds = 1.0;  // (psa_solver_desc::march_wait_us)

// The gate: a word that counts the workgroups that have started, with two flags.
// kGivenUp: a workgroup waited too long for the others to start, so none takes a
// step and k_march_alone takes them all. It is set only while some have not started
// (compare and swap on the word), and nobody passes before all have, so that
// every workgroup sees the same answer. kLost: a wait behind the gate took
// longer than any step can. Of more than kGateGroup workgroups every kGateGroup
// count in a line of their own and the last of them in the word: a line takes its
// additions one after the other.
constexpr unsigned int kGivenUp = 1u << 31;
constexpr unsigned int kLost = 1u << 30;
constexpr int kGateGroup = 16;
constexpr int kGateLine = 32;  // words of a line

constexpr int gate_groups(int tiles) {
  return tiles > kGateGroup ? (tiles + kGateGroup - 1) / kGateGroup : 0;
}
// Bytes of the gate.
constexpr size_t gate_bytes(int tiles) {
  return sizeof(unsigned int) * static_cast<size_t>(1 + kGateLine * gate_groups(tiles));
}

// Before the steps: words that no step waits for.
__global__ void k_march_init(unsigned long long *words, int nmax, int nall,
                             unsigned int *gate, unsigned int state, int groups) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < nall) words[i] = i < nmax ? kTurn : 0ull;
  if (i <= groups) gate[kGateLine * i] = i == 0 ? state : 0u;
}

template <typename T>
struct MarchArgs {
  const T *in;
  T *out;
  T *k1;  // k_march_alone's stage states (k2 holds the words and the gate until then)
  T *k2;
  Exchange<T> x;
  unsigned int *gate;
  long long nsteps;
  long long gate_ticks;  // limits of the waits at and behind the gate, in
  long long wait_ticks;  // wall-clock ticks
};

__device__ __forceinline__ unsigned int gate_state(const unsigned int *gate) {
  return __hip_atomic_load(gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The first half of counting a workgroup in (one thread), and the second, with
// the first one's result, which takes as long as a load.
template <typename T>
__device__ __forceinline__ unsigned int reach_gate(const MarchArgs<T> &f, int tile) {
  unsigned int *w = f.gate;
  if (f.x.tiles > kGateGroup) w += kGateLine * (1 + tile / kGateGroup);
  return __hip_atomic_fetch_add(w, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void count_group(const MarchArgs<T> &f, int tile,
                                            unsigned int before) {
  if (f.x.tiles <= kGateGroup) return;
  const int left = f.x.tiles - tile / kGateGroup * kGateGroup;
  if (static_cast<int>(before) + 1 == (left < kGateGroup ? left : kGateGroup))
    __hip_atomic_fetch_add(f.gate, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until every workgroup has started (one wave). False: given up.
template <typename T>
__device__ __forceinline__ bool pass_gate(const MarchArgs<T> &f, long long began) {
  const unsigned int all =
      static_cast<unsigned int>(f.x.tiles > kGateGroup ? gate_groups(f.x.tiles) : f.x.tiles);
  for (;;) {
    unsigned int g = gate_state(f.gate);
    if ((g & kGivenUp) != 0) return false;
    if ((g & ~kLost) == all) return true;
    if (wall_clock64() - began >= f.gate_ticks && (threadIdx.x & 63) == 0)
      __hip_atomic_compare_exchange_strong(f.gate, &g, g | kGivenUp, __ATOMIC_RELAXED,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Whether a wait that began then may go on (asked every kSpins loads: the flag's
// load would double the time between two looks at the words).
constexpr unsigned int kSpins = 256;

template <typename T>
__device__ __forceinline__ bool waits(const MarchArgs<T> &f, long long began) {
  return wall_clock64() - began < f.wait_ticks &&
         (gate_state(f.gate) & (kGivenUp | kLost)) == 0;
}

// What a call leaves in the control block (threads 0 .. 63): without a step the
// slots of the maximum stay as they are, for tiles that start later still read
// them, and a mixture of old and new ones could have them take a step that the
// others do not.
template <typename T>
__device__ __forceinline__ void march_control(psa_control *ctrl, int tid, bool from_state,
                                              bool taken, unsigned long long umax,
                                              unsigned long long umax_used, double t,
                                              long long mstep, int status, bool active,
                                              T dt_last) {
  if (from_state && taken) ctrl->umax_slot[tid][0] = tid == 0 ? umax : 0ull;
  if (tid != 0) return;
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
// Every workgroup has to be resident for the waits to end. The launch takes no
// more than a quarter of what the device holds (launch_march_cells), so that the
// marches of four streams fit together; where it still does not get its place (more
// of them, other processes, a stream with few CUs) the first exchange, whose gate
// they all have to reach, gives up for all after a second, before anything but the
// scratch array is written, and the launch behind it (k_march_alone) takes the
// steps. Behind the gate all are resident and stay so; a wait of ten minutes there
// ends the call with the status PSA_ERR_HIP.
//
// Bound by latency up to some 10^5 cells: the instructions of one wave, as in
// the ring schedule, and one exchange through memory (1.1 to 1.7 us), against a
// launch, load, control block and drain per step; above, by the FP64 rate of the
// few waves; the gate and the two launches beside it take some 3 us a call.
// FP64, Rusanov, WENO-JS5, us a step as a launch each and as a march:
// N = 1500 5.23, 2.58; 16384 5.05, 2.90; 47104 5.14, 3.30; 112640 5.47, 3.82;
// 243712 6.50, 4.81; 374784 7.46, 6.11; 505856 8.41, 7.18 (FP32 4.79, 2.44 to 6.55,
// 6.09). Lax-Friedrichs, as three launches a step and as a march: N = 184 12.9,
// 2.4; 16384 15.3, 6.1; 112640 15.7, 7.9; 505856 19.8, 11.1 (FP32 12.6, 2.1 to
// 17.5, 10.2). With learned weights the network's latency rules and both take the
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

  unsigned int before = 0;
  if (tid == 0 && tiles > 1) before = reach_gate(f, tile);
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

  bool given_up = false;
  if (tid == 0 && tiles > 1) count_group(f, tile, before);

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
    // tiles a wave); the first time, for every workgroup to have started (a
    // wave beside those two)
    const long long began = wall_clock64();
    bool ok = true;
    if (turns == 1 && wave == 1) ok = pass_gate(f, began);
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
    // everyone leaves
    given_up = (gate_state(f.gate) & kGivenUp) != 0;
    if (tid == 0 && !given_up)
      __hip_atomic_fetch_or(f.gate, kLost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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
      if (given_up) return;  // (with nothing written: k_march_alone's steps)
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
  if (tile == 0 && tid < 64)
    march_control<T>(ctrl, tid, from_state, taken, umax, umax_used, t, mstep, status, active,
                     dt_last);
}

// The steps of a march that was given up, by one workgroup (a launch behind every
// march of several tiles, which ends at once otherwise): stage sweeps over the
// state in memory with the march's arithmetic and decisions. It waits for nobody,
// so the steps are taken whatever else the device runs, though on one CU.
constexpr int kAloneBlock = 512;

template <typename T, int FLUX, int REC>
__global__ __launch_bounds__(kAloneBlock) void k_march_alone(StageArgs<T> p, MarchArgs<T> f) {
  if ((gate_state(f.gate) & kGivenUp) == 0) return;
  constexpr bool LF = FLUX == PSA_FLUX_LAX_FRIEDRICHS;
  constexpr int CPT = 2;
  constexpr int HALO = 3;  // of a stage
  constexpr int OUT = 64 * CPT - 2 * HALO;
  constexpr int WAVES = kAloneBlock / 64;
  __shared__ unsigned long long s_red[WAVES];
  psa_control *ctrl = p.ctrl;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = p.g;
  const int k0 = CPT * (tid & 63);
  const StepParams<T> par(ctrl);
  const bool from_state = ctrl->speed_from_state != 0;
  unsigned long long umax = gather_umax(ctrl);
  unsigned long long umax_used = umax;
  double t = ctrl->t;
  long long mstep = ctrl->m;
  int status = ctrl->status;
  bool active = false;
  bool taken = false;
  T dt_last = T(0), lam = T(0);
  StageArgs<T> pl = p;
  const MlpSource none{nullptr, nullptr};
  // (every thread has read the gate: the sweeps write over it)
  __syncthreads();

  // One stage of the whole state, and the maximum of |dst|: cells of a wave's
  // window but for three on either side; un may be dst.
  auto sweep = [&](int stage, const T *src, const T *un, T *dst) -> unsigned long long {
    T mx = T(0);
    bool nan = false;
    for (int64_t first = static_cast<int64_t>(wave) * OUT - HALO; first + HALO < p.n;
         first += WAVES * OUT) {
      const PeriodicSpan span(first + g, p.n, g);
      T x[CPT], dF[CPT];
#pragma unroll
      for (int r = 0; r < CPT; ++r) x[r] = span.load(src, k0 + r);
      wave_fluxes<T, FLUX, false, REC, CPT>(pl, x, dF, none, nullptr);
#pragma unroll
      for (int r = 0; r < CPT; ++r) {
        const int k = k0 + r;
        const int64_t i = first + k;
        if (k < HALO || k >= HALO + OUT || i >= p.n) continue;
        const T u = un[g + i];
        const T v = stage == 1   ? stage_value<T, 1>(x[r], u, lam, dF[r])
                    : stage == 2 ? stage_value<T, 2>(x[r], u, lam, dF[r])
                                 : stage_value<T, 3>(x[r], u, lam, dF[r]);
        dst[g + i] = v;
        mx = fmax(mx, fabs(v));
        nan |= isnan(v);
      }
    }
    mx = wave_max(mx);
    const bool any_nan = __any(nan);
    if ((tid & 63) == 63) s_red[wave] = any_nan ? nan_bits<T>() : abs_bits(mx);
    __syncthreads();
    unsigned long long top = s_red[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) top = s_red[w] > top ? s_red[w] : top;
    __syncthreads();
    return top;
  };

  const T *cur = f.in;
  for (long long s = 0; s < f.nsteps; ++s) {
    T dt = T(0);
    int st;
    umax_used = umax;
    active = control_decide_at<T>(par, t, mstep, status, umax, dt, st);
    status = st;
    if (__builtin_amdgcn_readfirstlane(active ? 1 : 0) == 0) break;
    lam = stage_lambda<T, FLUX>(p, dt);
    if constexpr (LF) pl.vconst = from_bits<T>(umax);
    unsigned long long top = sweep(1, cur, cur, f.k1);
    if constexpr (LF) pl.vconst = from_bits<T>(top);
    top = sweep(2, f.k1, cur, f.k2);
    if constexpr (LF) pl.vconst = from_bits<T>(top);
    top = sweep(3, f.k2, cur, f.out);
    if (from_state) umax = top;
    cur = f.out;
    t = static_cast<double>(static_cast<T>(t) + dt);
    mstep += 1;
    dt_last = dt;
    taken = true;
  }

  if (taken) {
    for (int k = tid; k < g; k += kAloneBlock) {
      f.out[k] = f.out[p.n + k];
      f.out[g + p.n + k] = f.out[g + k];
    }
  } else if (f.out != f.in) {
    for (int64_t c = tid; c < p.m; c += kAloneBlock) f.out[c] = f.in[c];
  }
  if (tid < 64)
    march_control<T>(ctrl, tid, from_state, taken, umax, umax_used, t, mstep, status, active,
                     dt_last);
}

// Cells of a workgroup with CPT cells per lane.
constexpr int march_cells(int cpt) { return kWaves * (64 * cpt - 2 * kHalo); }

template <typename T, int FLUX, int REC, int CPT>
int launch_march_cells(const StageArgs<T> &a, MarchArgs<T> f, void *scratch, hipStream_t s) {
  const int tiles =
      static_cast<int>((a.n + march_cells(CPT) - 1) / march_cells(CPT));
  const unsigned int resident = resident_blocks<k_march<T, FLUX, REC, CPT>>(kBlock);
  if (resident < 4u * static_cast<unsigned int>(tiles)) return PSA_ERR_NOT_IMPLEMENTED;
  // the exchange words and the gate in the caller's scratch array, in lines of
  // their own where there is room, else from the next multiple of 8 bytes on (the
  // arrays are aligned to 4 at least; no scratch: the caller asks whether it would
  // run)
  const int count = tiles > 1 ? Exchange<T>::count(tiles) : 0;
  const size_t need = sizeof(unsigned long long) * static_cast<size_t>(count) + gate_bytes(tiles);
  const size_t room = static_cast<size_t>(a.m) * sizeof(T);
  if (tiles > 1 && need + 4 > room) return PSA_ERR_NOT_IMPLEMENTED;
  const uintptr_t base = reinterpret_cast<uintptr_t>(scratch);
  uintptr_t at = (base + 127u) & ~static_cast<uintptr_t>(127);
  if (at - base + need > room) at = (base + 7u) & ~static_cast<uintptr_t>(7);
  if (scratch == nullptr) return PSA_OK;
  f.x.words = reinterpret_cast<unsigned long long *>(at);
  f.x.tiles = tiles;
  f.gate = reinterpret_cast<unsigned int *>(f.x.words + count);
  f.k2 = static_cast<T *>(scratch);
  if (tiles > 1) {
    hipLaunchKernelGGL(k_march_init, dim3(blocks_for(count, 256)), dim3(256), 0, s, f.x.words,
                       2 * tiles * Exchange<T>::SPREAD, count, f.gate,
                       f.gate_ticks < 0 ? kGivenUp : 0u, gate_groups(tiles));
    const int st = check_launch("march init");
    if (st != PSA_OK) return st;
  }
  hipLaunchKernelGGL((k_march<T, FLUX, REC, CPT>), dim3(static_cast<unsigned int>(tiles)),
                     dim3(kBlock), 0, s, a, f);
  const int st = check_launch("march steps");
  if (st != PSA_OK || tiles == 1) return st;
  hipLaunchKernelGGL((k_march_alone<T, FLUX, REC>), dim3(1), dim3(kAloneBlock), 0, s, a, f);
  return check_launch("march steps by one workgroup");
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
// against 21.5; FP64, N = 505856: 11.1 against 19.8).
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
                   void *k1, void *k2, hipStream_t s) {
  MarchArgs<T> f{};
  f.in = a.uk;
  f.out = a.out;
  f.k1 = static_cast<T *>(k1);
  f.nsteps = nsteps;
  int dev = 0, rate_khz = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess ||
      rate_khz <= 0) {
    (void)hipGetLastError();
    rate_khz = 100000;  // 100 MHz
  }
  f.wait_ticks = static_cast<long long>(kMarchWaitSeconds * 1000.0 * rate_khz);
  const double gate_s = d->march_wait_us != 0 ? 1.0e-6 * d->march_wait_us : kMarchGateSeconds;
  f.gate_ticks = gate_s < 0.0 ? -1 : static_cast<long long>(gate_s * 1000.0 * rate_khz);
  if (a.rec3) return launch_march_rec<T, 1>(d, a, f, k2, s);
  if (a.muscl) return launch_march_rec<T, 2>(d, a, f, k2, s);
  if (a.muscls) return launch_march_rec<T, 3>(d, a, f, k2, s);
  return launch_march_rec<T, 0>(d, a, f, k2, s);
}

}  // namespace
}  // namespace psa
