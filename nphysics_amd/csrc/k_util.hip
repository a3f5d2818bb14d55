// nphysics_amd/csrc/k_util.hip -- device-wide exclusive scan and stable LDS radix sort.
//
// Scan: one launch, 256-thread blocks each own a tile of 2048 words (8 per thread) and look back for
// the sum before it (scan.hpp). A launch per level (tiles, tile sums, add back) took 9-11 us above one
// tile, three dependent launches of 2.5-4 us each; now
// 3.4-5.8 us. Radix sort: 8-bit digits; per pass a histogram kernel (LDS
// atomics, one 256-bin row per tile, digit-major so that one exclusive scan yields every tile's
// output base) and a scatter kernel that ranks keys stably inside a tile with 64-lane wavefront
// ballots (eight ballots give each lane the set of lanes holding the same digit).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "scan.hpp"

namespace nph {

namespace {

constexpr int kScanItems = kScanTile / kScanThreads;

constexpr int kRadixThreads = 256;
constexpr int kRadixItems = 8;
constexpr int kRadixTile = kRadixThreads * kRadixItems;
constexpr int kRadixBins = 256;

__global__ void __launch_bounds__(kScanThreads) k_scan(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                                      int n, ScanRun run) {
  __shared__ uint32_t s_wave[kScanWaves];
  __shared__ uint32_t s_tile, s_before;
  const uint32_t tile = scan_tile(run, &s_tile);
  if (tile >= gridDim.x) return;  // only after a launch that failed: its tickets were never taken
  const long base = long(tile) * kScanTile + long(threadIdx.x) * kScanItems;
  uint32_t v[kScanItems];
  uint32_t acc = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    v[k] = base + k < n ? in[base + k] : 0u;
    acc += v[k];
  }
  uint32_t total;
  uint32_t at = block_exclusive(acc, s_wave, total);
  if (threadIdx.x < 64) {
    const uint32_t before = scan_look_back(run, tile, total);
    if (threadIdx.x == 0) s_before = before;
  }
  __syncthreads();
  at += s_before;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    if (base + k < n) out[base + k] = at;
    at += v[k];
  }
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, size_t n) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void __launch_bounds__(kRadixThreads) k_radix_hist(const uint32_t* __restrict__ keys,
                                                             int n, int shift, int ntiles,
                                                             uint32_t* __restrict__ hist) {
  __shared__ uint32_t s_h[kRadixBins];
  const int tid = threadIdx.x;
  s_h[tid] = 0;
  __syncthreads();
  const long base = long(blockIdx.x) * kRadixTile;
#pragma unroll
  for (int it = 0; it < kRadixItems; ++it) {
    const long i = base + it * kRadixThreads + tid;
    if (i < n) atomicAdd(&s_h[(keys[i] >> shift) & 255u], 1u);
  }
  __syncthreads();
  hist[long(tid) * ntiles + blockIdx.x] = s_h[tid];
}

__global__ void __launch_bounds__(kRadixThreads) k_radix_scatter(
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin, uint32_t* __restrict__ kout,
    uint32_t* __restrict__ vout, int n, int shift, int ntiles, const uint32_t* __restrict__ offs) {
  __shared__ uint32_t s_base[kRadixBins];
  __shared__ uint32_t s_wcnt[kRadixThreads / 64][kRadixBins];
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  s_base[tid] = offs[long(tid) * ntiles + blockIdx.x];
  const long base = long(blockIdx.x) * kRadixTile;
  for (int it = 0; it < kRadixItems; ++it) {
#pragma unroll
    for (int w = 0; w < kRadixThreads / 64; ++w) s_wcnt[w][tid] = 0;
    __syncthreads();
    const long i = base + it * kRadixThreads + tid;
    const bool valid = i < n;
    const uint32_t key = valid ? kin[i] : 0u;
    const uint32_t d = (key >> shift) & 255u;
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t bb = __ballot(bit);
      m &= bit ? bb : ~bb;
    }
    const uint32_t lrank = __popcll(m & lt_mask);
    if (valid && lrank == 0) s_wcnt[wave][d] = uint32_t(__popcll(m));
    __syncthreads();
    if (valid) {
      uint32_t pre = 0;
      for (int w = 0; w < wave; ++w) pre += s_wcnt[w][d];
      const uint32_t pos = s_base[d] + pre + lrank;
      kout[pos] = key;
      vout[pos] = vin[i];
    }
    __syncthreads();
    uint32_t tot = 0;
#pragma unroll
    for (int w = 0; w < kRadixThreads / 64; ++w) tot += s_wcnt[w][tid];
    s_base[tid] += tot;
    __syncthreads();
  }
}

int div_up(long a, long b) { return int((a + b - 1) / b); }

}  // namespace

ScanState::~ScanState() {
  if (mem) (void)hipFree(mem);
}

hipError_t ScanState::ensure(size_t need, hipStream_t s) {
  if (need <= tiles) return hipSuccess;
  const size_t grown = std::max(need + need / 2, size_t(1024));
  hipError_t e = hipStreamSynchronize(s);
  if (e != hipSuccess) return e;
  void* q = nullptr;
  if ((e = hipMalloc(&q, 64 + grown * sizeof(unsigned long long))) != hipSuccess) return e;
  if (mem) (void)hipFree(mem);
  mem = q;
  tiles = grown;
  base = epoch = 0;
  fill_u32(static_cast<uint32_t*>(mem), 0u, 16 + 2 * tiles, s);
  return hipSuccess;
}

ScanRun ScanState::next(uint32_t ntiles, hipStream_t s) {
  if (++epoch >= (1u << 30)) {  // the epochs start over on cleared words
    fill_u32(static_cast<uint32_t*>(mem) + 16, 0u, 2 * tiles, s);
    epoch = 1;
  }
  ScanRun r;
  r.ticket = static_cast<uint32_t*>(mem);
  r.word = reinterpret_cast<unsigned long long*>(static_cast<char*>(mem) + 64);
  r.base = base;
  r.epoch = epoch;
  base += ntiles;
  return r;
}

void scan_exclusive_u32(const uint32_t* in, uint32_t* out, int n, ScanState& st, hipStream_t s) {
  if (n <= 0) return;
  const uint32_t tiles = uint32_t(scan_tiles(size_t(n)));
  hipLaunchKernelGGL(k_scan, dim3(tiles), dim3(kScanThreads), 0, s, in, out, n, st.next(tiles, s));
}

size_t radix_temp_words(int n) {
  const int ntiles = div_up(n > 0 ? n : 1, kRadixTile);
  const size_t h = size_t(kRadixBins) * ntiles;
  return 2 * h;
}

size_t radix_scan_tiles(int n) { return scan_tiles(size_t(kRadixBins) * div_up(n > 0 ? n : 1, kRadixTile)); }

void radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt,
                      int n, int bits, uint32_t* tmp, ScanState& st, hipStream_t s) {
  if (n <= 1) return;
  const int ntiles = div_up(n, kRadixTile);
  const size_t h = size_t(kRadixBins) * ntiles;
  uint32_t* hist = tmp;
  uint32_t* offs = tmp + h;
  uint32_t* kin = keys;
  uint32_t* vin = vals;
  uint32_t* kout = keys_alt;
  uint32_t* vout = vals_alt;
  int passes = 0;
  for (int shift = 0; shift < bits; shift += 8, ++passes) {
    hipLaunchKernelGGL(k_radix_hist, dim3(ntiles), dim3(kRadixThreads), 0, s, kin, n, shift, ntiles, hist);
    scan_exclusive_u32(hist, offs, int(h), st, s);
    hipLaunchKernelGGL(k_radix_scatter, dim3(ntiles), dim3(kRadixThreads), 0, s, kin, vin, kout, vout, n,
                       shift, ntiles, offs);
    uint32_t* t = kin; kin = kout; kout = t;
    t = vin; vin = vout; vout = t;
  }
  if (passes & 1) {
    (void)hipMemcpyAsync(keys, kin, size_t(n) * 4, hipMemcpyDeviceToDevice, s);
    (void)hipMemcpyAsync(vals, vin, size_t(n) * 4, hipMemcpyDeviceToDevice, s);
  }
}

void fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_fill_u32, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, p, v, n);
}

}  // namespace nph
