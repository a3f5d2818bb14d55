// nphysics_amd/csrc/kernels.hpp -- launch wrappers of the HIP kernels (host side).
//
// Every wrapper enqueues on the given stream and returns immediately. Device pointers only.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace nph {

// ---------------------------------------------------------------- utilities (k_util.hip)
// One prefix sum's share of a world's scan state, passed to its kernel by value (scan.hpp).
struct ScanRun {
  unsigned long long* word;  // [tiles]
  uint32_t* ticket;
  uint32_t base, epoch;
};

// A world's scan state: the published words of up to `tiles` tiles and the ticket counter, both
// zeroed when made, and how far counter and epochs have come. One stream at a time uses it.
struct ScanState {
  void* mem = nullptr;  // ticket word, then the tile words at +64
  size_t tiles = 0;
  uint32_t base = 0, epoch = 0;

  ScanState() = default;
  ScanState(const ScanState&) = delete;
  ScanState& operator=(const ScanState&) = delete;
  ~ScanState();
  // Room for `need` tiles (grows by a new zeroed buffer, after the work on `s` has ended).
  hipError_t ensure(size_t need, hipStream_t s);
  // The next scan of `ntiles` workgroups, all of which take a ticket.
  ScanRun next(uint32_t ntiles, hipStream_t s);
};

// Exclusive prefix sum of n uint32 values, one launch; `st` must hold scan_tiles(n) tiles.
constexpr int kScanTile = 2048;
inline size_t scan_tiles(size_t n) { return (n + kScanTile - 1) / kScanTile; }
void scan_exclusive_u32(const uint32_t* in, uint32_t* out, int n, ScanState& st, hipStream_t s);

// Stable LSD radix sort of (key, value) pairs on the low `bits` bits of the key.
// Result ends in (keys, vals); (keys_alt, vals_alt) are scratch of the same size.
// `tmp` must hold radix_temp_words(n) words and `st` radix_scan_tiles(n) tiles.
size_t radix_temp_words(int n);
size_t radix_scan_tiles(int n);
void radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt,
                      int n, int bits, uint32_t* tmp, ScanState& st, hipStream_t s);

void fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s);

}  // namespace nph
