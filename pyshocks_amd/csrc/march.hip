// The march schedule: all the steps of a psa_ssprk33_steps call on a mid-size
// periodic state in one launch, a tile per workgroup held in LDS throughout.
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
constexpr int kHalo = 9;       // cells a step reads on either side of a tile
constexpr int kMargin = 12;    // first own cell of a tile in its LDS layout
constexpr int kMarchMaxTiles = 256;
constexpr double kMarchWaitSeconds = 600.0;

// What the tiles hand each other after a step, in words of 64 bits that are
// stored and loaded whole and say themselves which step they are of, so that
// no order between them is needed: per tile max|u| of its new cells, the parity
// of the step's turn in the (free) sign bit, and its first and last 9 cells, 32
// bits a word under the step's number. Two sets, used in turn: a tile writes a
// set again only after it has read every tile's words of the step in between,
// which each tile writes after it is done with that set. The words are spread
// over the lines (two maxima to a line, the edges in lines of their own): a
// line takes its writes one after the other, and with the maxima packed 16 to a
// line an exchange of 69 tiles took 2.4 us instead of 1.15.
template <typename T>
struct Exchange {
  static constexpr int NW = sizeof(T) / 4;          // words per cell
  static constexpr int SIDE = kHalo * NW;           // words per side
  static constexpr int PAD = (SIDE + 15) / 16 * 16; // in whole lines of 128 bytes
  static constexpr int SPREAD = 8;                  // words from maximum to maximum
  unsigned long long *words;
  int tiles;

  __device__ __forceinline__ unsigned long long *max_word(int set, int tile) const {
    return words + (set * tiles + tile) * SPREAD;
  }
  // side 0: the first cells of the tile, side 1: the last ones
  __device__ __forceinline__ unsigned long long *cells(int set, int tile, int side) const {
    return words + 2 * tiles * SPREAD + ((set * tiles + tile) * 2 + side) * PAD;
  }
  static int count(int tiles) { return tiles * (2 * SPREAD + 4 * PAD); }
};

__device__ __forceinline__ void put(unsigned long long *w, unsigned long long v) {
  __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long get(const unsigned long long *w) {
  return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

constexpr unsigned long long kTurn = 1ull << 63;

__device__ __forceinline__ unsigned int word_of(float v, int) { return __float_as_uint(v); }
__device__ __forceinline__ unsigned int word_of(double v, int k) {
  return static_cast<unsigned int>(k == 0 ? __double2loint(v) : __double2hiint(v));
}

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
// every value in between are the whole-step schedule's bit for bit. Workgroup b
// holds the cells [b n / G, (b + 1) n / G) and 12 on either side in
// step_tile's layout; after a step it publishes its new maximum and edge cells
// and waits for every tile's maximum and its neighbours' edges.
//
// Every workgroup has to be resident for the waits to end: the launch takes no
// more than a quarter of what the device holds (launch_march_cells), so that the
// marches of four streams fit together, kernels that end by themselves only delay
// it, and a wait of ten minutes gives up for all (status PSA_ERR_HIP).
//
// Bound by latency: the three stages (1.65 us with one cell per thread) and one
// exchange through memory, against a launch, load, control block and drain per
// step. FP64, Rusanov, us a step as a launch each and as a march: N = 2000 4.73,
// 2.71; 16384 4.98, 2.81; 61000 5.19, 3.41; 131072 5.98, 4.52; 258000 6.83, 5.03
// (FP32 4.55, 2.54 to 5.71, 4.19). With learned weights the network's latency
// rules and both take the same, so they stay on the step kernel.
template <typename T, int FLUX, int VEL, int CPT, int REC>
__global__ __attribute__((amdgpu_flat_work_group_size(1, kBlock),
                          amdgpu_waves_per_eu(4))) void k_march(StageArgs<T> p, MarchArgs<T> f) {
  using SM = StepSmem<T, kBlock, CPT, FLUX == PSA_FLUX_ESWENO>;
  using X = Exchange<T>;
  constexpr int C = SM::C;
  constexpr int L = SM::L;
  constexpr int WAVES = kBlock / 64;
  __shared__ SM sm;
  __shared__ unsigned long long s_max[WAVES];
  __shared__ int s_abort;
  psa_control *ctrl = p.ctrl;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = p.g;
  const int tiles = f.x.tiles;
  const int tile = static_cast<int>(blockIdx.x);
  const int64_t start = p.n * tile / tiles;
  const int cnt = static_cast<int>(p.n * (tile + 1) / tiles - start);
  const int left = tile == 0 ? tiles - 1 : tile - 1;
  const int right = tile == tiles - 1 ? 0 : tile + 1;

  {
    const PeriodicSpan span(start + g - kMargin, p.n, g);
    for (int j = tid; j < L; j += kBlock) sm.x0[j] = span.load(f.in, j);
  }
  // entries without a neighbouring thread (outside the exact ranges)
  if (tid < 8) sm.x1[tid < 4 ? tid : C + tid] = T(0);
  if (tid == 0) {
    sm.urL[0] = T(0);
    sm.ulF[kBlock] = T(0);
    if constexpr (FLUX == PSA_FLUX_ESWENO) {
      sm.omL[0] = T(0);
      sm.omR[kBlock] = T(0);
    }
    s_abort = 0;
  }
  const StepParams<T> par(ctrl);
  const bool from_state = ctrl->speed_from_state != 0;
  unsigned long long umax = gather_umax(ctrl);
  unsigned long long umax_used = umax;  // max|u| of the last decision
  double t = ctrl->t;
  long long mstep = ctrl->m;
  int status = ctrl->status;
  bool active = false;
  bool taken = false;
  T dt_last = T(0);
  __syncthreads();

  const int j0 = 4 + CPT * tid;
  T un[CPT], val[CPT];
#pragma unroll
  for (int r = 0; r < CPT; ++r) un[r] = val[r] = sm.x0[j0 + r];
  const MlpSource none{nullptr, nullptr};
  for (long long s = 0; s < f.nsteps; ++s) {
    T dt = T(0);
    int st;
    umax_used = umax;
    active = control_decide_at<T>(par, t, mstep, status, umax, dt, st);
    status = st;
    if (!active) break;  // the same in every workgroup
    step_stage<T, FLUX, VEL, kBlock, CPT, 1, false, REC>(p, sm.x0, sm, dt, un, val, none, nullptr);
#pragma unroll
    for (int r = 0; r < CPT; ++r) sm.x1[j0 + r] = val[r];
    __syncthreads();
    step_stage<T, FLUX, VEL, kBlock, CPT, 2, false, REC>(p, sm.x1, sm, dt, un, val, none, nullptr);
#pragma unroll
    for (int r = 0; r < CPT; ++r) sm.x0[j0 + r] = val[r];
    __syncthreads();
    step_stage<T, FLUX, VEL, kBlock, CPT, 3, false, REC>(p, sm.x0, sm, dt, un, val, none, nullptr);
    t = static_cast<double>(static_cast<T>(t) + dt);
    mstep += 1;
    dt_last = dt;
    taken = true;

    // ---- publish the edges, then the maximum (every read of x0 ended before
    // the exchange barrier of stage 3)
    const int set = static_cast<int>(s & 1);
    const unsigned long long tag = static_cast<unsigned long long>(
                                       static_cast<unsigned int>(s + 1))
                                   << 32;
    const unsigned long long turn = (s & 2) != 0 ? kTurn : 0ull;
    T mx = T(0);
    bool nan = false;
#pragma unroll
    for (int r = 0; r < CPT; ++r) {
      const int o = j0 + r - kMargin;  // own cell
      if (o >= 0 && o < cnt) {
        sm.x0[j0 + r] = val[r];
        mx = fmax(mx, fabs(val[r]));
        nan |= isnan(val[r]);
        if (o < kHalo) {
          unsigned long long *w = f.x.cells(set, tile, 0) + X::NW * o;
#pragma unroll
          for (int k = 0; k < X::NW; ++k) put(w + k, tag | word_of(val[r], k));
        }
        if (o >= cnt - kHalo) {
          unsigned long long *w = f.x.cells(set, tile, 1) + X::NW * (o - (cnt - kHalo));
#pragma unroll
          for (int k = 0; k < X::NW; ++k) put(w + k, tag | word_of(val[r], k));
        }
      }
    }
    const unsigned long long wmax = wave_max_u64(nan ? nan_bits<T>() : abs_bits(mx));
    if (lane == 0) sm.red[wave] = wmax;
    __syncthreads();
    if (tid == 0) {
      unsigned long long v = sm.red[0];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) v = sm.red[w] > v ? sm.red[w] : v;
      put(f.x.max_word(set, tile), turn | v);
    }

    // ---- wait for the neighbours' edges (the last wave) and every maximum
    // (64 tiles a wave)
    const long long began = wall_clock64();
    bool ok = true;
    unsigned long long top = 0;
    if (wave == WAVES - 1) {
      const bool mine = lane < 2 * X::SIDE;
      const int side = lane < X::SIDE ? 0 : 1;
      const int k = lane - side * X::SIDE;
      // the cells left of the tile are the left tile's last ones
      const unsigned long long *w =
          mine ? f.x.cells(set, side == 0 ? left : right, side == 0 ? 1 : 0) + k : nullptr;
      unsigned long long v = tag;
      for (unsigned int spin = 1;; ++spin) {
        if (mine) v = get(w);
        const bool there = (v & 0xFFFFFFFF00000000ull) == tag;
        if (__all(there)) break;
        if (spin % kSpins == 0 && !(ok = waits(f, began))) break;
      }
      const unsigned int bits = static_cast<unsigned int>(v);
      // own cells start at kMargin: the halo cells are the 9 before and behind
      const int at = side == 0 ? kMargin - kHalo : kMargin + cnt;
      if constexpr (X::NW == 2) {
        const unsigned int hi = __shfl_down(bits, 1, 64);
        if (mine && (k & 1) == 0)
          sm.x0[at + (k >> 1)] = __hiloint2double(static_cast<int>(hi), static_cast<int>(bits));
      } else {
        if (mine) sm.x0[at + k] = __uint_as_float(bits);
      }
    }
    for (int first = 64 * wave; first < tiles; first += kBlock) {
      const bool mine = first + lane < tiles;
      const unsigned long long *w = f.x.max_word(set, first + lane);
      unsigned long long v = turn;
      for (unsigned int spin = 1; ok; ++spin) {
        if (mine) v = get(w);
        if (__all((v & kTurn) == turn)) break;
        if (spin % kSpins == 0) ok = waits(f, began);
      }
      v &= ~kTurn;
      top = v > top ? v : top;
    }
    top = wave_max_u64(top);
    if (lane == 0) {
      s_max[wave] = top;
      if (!ok) s_abort = 1;
    }
    __syncthreads();
    if (s_abort != 0) {
      // a workgroup is not running: everyone leaves
      if (tid == 0) __hip_atomic_store(f.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      status = PSA_ERR_HIP;
      break;
    }
    if (from_state) {
      umax = s_max[0];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) umax = s_max[w] > umax ? s_max[w] : umax;
    }
#pragma unroll
    for (int r = 0; r < CPT; ++r) un[r] = sm.x0[j0 + r];
  }

  // ---- the tile's cells and their ghost images
  if (taken || f.out != f.in) {
    for (int o = tid; o < cnt; o += kBlock) {
      const T v = sm.x0[kMargin + o];
      const int64_t i = start + o;
      f.out[g + i] = v;
      if (taken) {
        if (i < g) f.out[g + p.n + i] = v;
        if (i >= p.n - g) f.out[g + i - p.n] = v;
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

// The smallest tiles that leave a march within kMarchMaxTiles workgroups.
int march_cells_per_thread(int64_t n) {
  for (int cpt = 1; cpt <= 4; cpt *= 2) {
    if (n <= static_cast<int64_t>(kMarchMaxTiles) * (kBlock * cpt - 16)) return cpt;
  }
  return 0;
}

template <typename T, int FLUX, int VEL, int CPT, int REC>
int launch_march_cells(const StageArgs<T> &a, MarchArgs<T> f, void *scratch, hipStream_t s) {
  constexpr int TO = kBlock * CPT - 16;
  // (evenly split: n / tiles is at least TO / 2 here, far more than the margins)
  const int tiles = static_cast<int>((a.n + TO - 1) / TO);
  auto kernel = k_march<T, FLUX, VEL, CPT, REC>;
  const unsigned int resident =
      resident_blocks<k_march<T, FLUX, VEL, CPT, REC>>(kBlock);
  if (resident < 4u * static_cast<unsigned int>(tiles)) return PSA_ERR_NOT_IMPLEMENTED;
  // the exchange words and the abort flag in the caller's scratch array
  const uintptr_t at =
      (reinterpret_cast<uintptr_t>(scratch) + 127u) & ~static_cast<uintptr_t>(127);
  const int count = Exchange<T>::count(tiles);
  const size_t need = sizeof(unsigned long long) * static_cast<size_t>(count) + sizeof(int) +
                      (at - reinterpret_cast<uintptr_t>(scratch));
  if (need > static_cast<size_t>(a.m) * sizeof(T)) return PSA_ERR_NOT_IMPLEMENTED;
  f.x.words = reinterpret_cast<unsigned long long *>(at);
  f.x.tiles = tiles;
  f.abort = reinterpret_cast<int *>(f.x.words + count);
  hipLaunchKernelGGL(k_march_init, dim3(blocks_for(count, 256)), dim3(256), 0, s, f.x.words,
                     2 * tiles * Exchange<T>::SPREAD, count, f.abort);
  int st = check_launch("march init");
  if (st != PSA_OK) return st;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned int>(tiles)), dim3(kBlock), 0, s, a, f);
  return check_launch("march steps");
}

template <typename T, int FLUX, int VEL, int REC>
int launch_march_tiles(const StageArgs<T> &a, const MarchArgs<T> &f, void *scratch,
                       hipStream_t s) {
  switch (march_cells_per_thread(a.n)) {
    case 1:
      return launch_march_cells<T, FLUX, VEL, 1, REC>(a, f, scratch, s);
    case 2:
      return launch_march_cells<T, FLUX, VEL, 2, REC>(a, f, scratch, s);
    case 4:
      return launch_march_cells<T, FLUX, VEL, 4, REC>(a, f, scratch, s);
    default:
      return PSA_ERR_NOT_IMPLEMENTED;
  }
}

template <typename T, int REC>
int launch_march_rec(const psa_solver_desc *d, const StageArgs<T> &a, const MarchArgs<T> &f,
                     void *scratch, hipStream_t s) {
  if (d->flux == PSA_FLUX_RUSANOV)
    return launch_march_tiles<T, PSA_FLUX_RUSANOV, 0, REC>(a, f, scratch, s);
  if (d->flux == PSA_FLUX_BURGERS_UPWIND)
    return launch_march_tiles<T, PSA_FLUX_BURGERS_UPWIND, 0, REC>(a, f, scratch, s);
  if (d->flux == PSA_FLUX_ENGQUIST_OSHER)
    return launch_march_tiles<T, PSA_FLUX_ENGQUIST_OSHER, 0, REC>(a, f, scratch, s);
  if constexpr (REC == 1) {
    if (d->flux == PSA_FLUX_ESWENO)
      return launch_march_tiles<T, PSA_FLUX_ESWENO, 0, REC>(a, f, scratch, s);
  }
  return launch_march_tiles<T, PSA_FLUX_ADVECTION_UPWIND, 1, REC>(a, f, scratch, s);
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

int launch_march(const psa_solver_desc *d, const StageArgs<double> &a, long long nsteps,
                 void *scratch, hipStream_t s) {
  return launch_march_t<double>(d, a, nsteps, scratch, s);
}
int launch_march(const psa_solver_desc *d, const StageArgs<float> &a, long long nsteps,
                 void *scratch, hipStream_t s) {
  return launch_march_t<float>(d, a, nsteps, scratch, s);
}

}  // namespace psa
