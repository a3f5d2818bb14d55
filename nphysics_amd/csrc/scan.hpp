// nphysics_amd/csrc/scan.hpp -- device side of the one-launch prefix sums (k_util.hip and the
// kernels that scan what they compute).
//
// Decoupled look-back (Merrill and Garland, 2016): tiles take their numbers from a ticket counter, each
// publishes its own sum as soon as it has it and then its inclusive prefix, and one wave of a tile
// reads 64 predecessors at a time until it meets a prefix. A number taken by ticket means that every
// lower-numbered tile has begun and publishes without waiting for anyone, so the wait ends. A
// published word holds value, epoch and state together and is moved by one relaxed 64-bit atomic, so
// no fence (on this card an L2 write-back across the eight dies) is needed; the epoch, one per scan,
// makes words of earlier scans read as "not there yet" and saves clearing them.
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace nph {

constexpr int kScanThreads = 256;
constexpr int kScanWaves = kScanThreads / 64;

__device__ __forceinline__ uint32_t wave_inclusive(uint32_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t x = __shfl_up(v, off);
    if (lane >= off) v += x;
  }
  return v;
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Exclusive prefix of v over a workgroup of kScanThreads lanes; `total` receives the sum.
// s_wave: kScanWaves words. Every lane of the workgroup calls it; ends with a barrier.
__device__ __forceinline__ uint32_t block_exclusive(uint32_t v, uint32_t* s_wave, uint32_t& total) {
  const int wave = threadIdx.x >> 6;
  const uint32_t inc = wave_inclusive(v);
  if ((threadIdx.x & 63) == 63) s_wave[wave] = inc;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kScanWaves; ++w) {
    const uint32_t x = s_wave[w];
    if (w < wave) before += x;
    all += x;
  }
  total = all;
  __syncthreads();
  return before + inc - v;
}

// This workgroup's tile number. s_tile: one word. Ends with a barrier.
__device__ __forceinline__ uint32_t scan_tile(const ScanRun& r, uint32_t* s_tile) {
  if (threadIdx.x == 0) *s_tile = atomicAdd(r.ticket, 1u) - r.base;
  __syncthreads();
  const uint32_t t = *s_tile;
  __syncthreads();
  return t;
}

__device__ __forceinline__ unsigned long long scan_word(uint32_t value, uint32_t epoch, uint32_t state) {
  return (static_cast<unsigned long long>(value) << 32) | (epoch << 2) | state;
}

// Publishes tile's sum and returns the sum of all tiles before it. Called by all 64 lanes of one wave.
__device__ __forceinline__ uint32_t scan_look_back(const ScanRun& r, uint32_t tile, uint32_t sum) {
  const int lane = threadIdx.x & 63;
  if (lane == 0)
    __hip_atomic_store(r.word + tile, scan_word(sum, r.epoch, tile == 0 ? 2u : 1u), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  if (tile == 0) return 0u;
  uint32_t before = 0;
  for (int top = int(tile) - 1;; top -= 64) {
    const int t = top - lane;
    unsigned long long w = scan_word(0u, r.epoch, 2u);
    for (;;) {
      if (t >= 0) w = __hip_atomic_load(r.word + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool there = (uint32_t(w) >> 2) == r.epoch && (uint32_t(w) & 3u) != 0u;
      if (__all(there)) break;
      __builtin_amdgcn_s_sleep(1);
    }
    const uint64_t full = __ballot((uint32_t(w) & 3u) == 2u);
    const int last = full ? __ffsll(static_cast<long long>(full)) - 1 : 63;
    before += wave_sum(lane <= last ? uint32_t(w >> 32) : 0u);
    if (full) break;
  }
  if (lane == 0)
    __hip_atomic_store(r.word + tile, scan_word(before + sum, r.epoch, 2u), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  return before;
}

}  // namespace nph
