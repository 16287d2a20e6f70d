// Exchange of edge cells and maxima between workgroups of one launch.
#pragma once

#include <hip/hip_runtime.h>

#include "wave_device.hpp"

namespace psa {

// What workgroups with a tile of a state each hand each other after a step, in
// words of 64 bits that are stored and loaded whole and say themselves which step
// they are of, so that no order between them (no fence, no write-back of a
// cache) is needed: per tile max|u| of its new cells, the parity
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
  static constexpr int SIDE = kWaveHalo * NW;           // words per side
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
  static constexpr int count(int tiles) { return tiles * (2 * SPREAD + 4 * PAD); }
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

}  // namespace psa
