// nphysics_amd/csrc/k_narrowphase.hip -- narrow phase: one lane per broad-phase pair.
//
// Replaces GeometricalWorld::perform_narrow_phase (src/world/geometrical_world.rs:315-320) over
// the interaction graph and the manifold collection of MechanicalWorld::step
// (src/world/mechanical_world.rs:287-300, manifolds with at least one contact). Each lane runs the
// contact generator of its pair (np_geometry.hpp) with prediction = sum of both query limits and
// writes up to 4 contacts as 96-byte records into the pair's fixed slots, where they stay; a scan
// then lists the manifolds (pairs with contacts, in pair order) with their first slot and count.
// The contact order (pair order, then generator order) is the manifold list's. HBM bound: 100 B
// per pair + 48 B per contact of algorithmic traffic.
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "np_geometry.hpp"
#include "scan.hpp"
#include "stages.hpp"

namespace nph {

namespace {

// Lanes are binned by pair kind: cuboid-cuboid pairs (SAT + clipping, the expensive one) are run by
// k_np_boxes with their clip polygons in LDS, all other pairs by k_np_balls. The compaction of the
// broad phase fills the two lists as it writes the pairs; k_np_bin does it for lists of pairs from
// elsewhere. The order within a list is arbitrary: every pair writes its own slots.
__global__ void __launch_bounds__(256) k_np_bin(DevBodies b, const int2* __restrict__ pairs, NarrowPhaseBufs np,
                                               DevContacts out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (out.bfirst && i < out.bcount) out.bfirst[i] = -1;
  const bool in = i < int(*np.npairs);
  bool box = false;
  if (in) {
    const int2 pr = pairs[i];
    box = b.shape[pr.x] == SHAPE_CUBOID && b.shape[pr.y] == SHAPE_CUBOID;
  }
  const uint64_t mb = __ballot(in && box), ma = __ballot(in && !box);
  const int lane = threadIdx.x & 63;
  uint32_t wb = 0, wa = 0;
  if (lane == 0) {
    if (mb) wb = atomicAdd(np.nbox, uint32_t(__popcll(mb)));
    if (ma) wa = atomicAdd(np.nball, uint32_t(__popcll(ma)));
  }
  wb = __shfl(wb, 0);
  wa = __shfl(wa, 0);
  const uint64_t below = (1ull << lane) - 1ull;
  if (in && box) np.perm[wb + uint32_t(__popcll(mb & below))] = uint32_t(i);
  if (in && !box) np.perm[uint32_t(np.pair_cap) - 1u - (wa + uint32_t(__popcll(ma & below)))] = uint32_t(i);
}

// Writes contact k of pair i as a 96-byte record into the pair's slots.
__device__ __forceinline__ void put_contact(const DevContacts& out_c, int i, int k, const Contact& ct) {
  float4* r = out_c.contact(long(i) * kPairSlots + k);
  r[0] = f4(ct.w1, ct.depth);
  r[1] = f4(ct.w2, __uint_as_float(ct.feature));
  r[2] = f4(ct.n, __int_as_float(ct.kind));
  r[3] = f4(ct.lp1, 0.0f);
  r[4] = f4(ct.lp2, 0.0f);
  r[5] = f4(ct.ln, 0.0f);
}

// Cuboid-cuboid pairs: SAT + clipping, the clip polygons
// and separations of each lane interleaved in LDS.
constexpr int kBoxBlock = 64;
__global__ void __launch_bounds__(kBoxBlock) k_np_boxes(DevBodies b, const int2* __restrict__ pairs,
                                                       NarrowPhaseBufs np, DevContacts out_c) {
  __shared__ ClipVert s_poly[2 * 8 * kBoxBlock];
  __shared__ float s_sep[8 * kBoxBlock];
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= int(*np.nbox)) return;
  const int i = int(np.perm[j]);
  const int2 pr = pairs[i];
  const int a = pr.x, c = pr.y;
  const float prediction = b.qlim[a] + b.qlim[c];
  const PolyBuf p0{s_poly + threadIdx.x, kBoxBlock}, p1{s_poly + 8 * kBoxBlock + threadIdx.x, kBoxBlock};
  const SepBuf sep{s_sep + threadIdx.x, kBoxBlock};
  const int nc = collide_box_box(xyz(b.pos(a)), toq(b.rot(a)), xyz(b.dims[a]), xyz(b.pos(c)), toq(b.rot(c)),
                                 xyz(b.dims[c]), prediction, p0, p1, sep,
                                 [&](int k, const Contact& ct) { put_contact(out_c, i, k, ct); });
  np.count[i] = uint32_t(nc);
}

// Pairs with a ball.
__global__ void __launch_bounds__(256) k_np_balls(DevBodies b, const int2* __restrict__ pairs, NarrowPhaseBufs np,
                                                 DevContacts out_c) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= int(*np.nball)) return;
  const int i = int(np.perm[np.pair_cap - 1 - j]);
  const int2 pr = pairs[i];
  const int a = pr.x, c = pr.y;
  const float prediction = b.qlim[a] + b.qlim[c];
  const int nc = collide_ball_pair(b.shape[a], xyz(b.dims[a]), xyz(b.pos(a)), toq(b.rot(a)), b.shape[c],
                                   xyz(b.dims[c]), xyz(b.pos(c)), toq(b.rot(c)), prediction,
                                   [&](int k, const Contact& ct) { put_contact(out_c, i, k, ct); });
  np.count[i] = uint32_t(nc);
}

// The manifold list: one entry per pair with contacts, in pair order (its contacts stay in the pair's
// slots), and per body the first manifold it is body 1 of. One launch: each workgroup's tile of
// pairs looks back for the manifolds before it (scan.hpp). The scans of flags and counts, the list
// and the index were eight launches of 2.5-4 us: 30 us and more together, now
// 4.7 us at 3,566 pairs and 13 us at 533,260.
constexpr int kManifoldItems = 8;
constexpr int kManifoldTile = kScanThreads * kManifoldItems;

__global__ void __launch_bounds__(kScanThreads) k_np_manifolds(const int2* __restrict__ pairs, NarrowPhaseBufs np,
                                                              DevContacts out, ScanRun run) {
  __shared__ uint32_t s_wave[kScanWaves];
  __shared__ uint32_t s_tile, s_before;
  const uint32_t tile = scan_tile(run, &s_tile);
  if (tile >= gridDim.x) return;  // only after a launch that failed: its tickets were never taken
  const int npairs = int(*np.npairs) < np.pair_cap ? int(*np.npairs) : np.pair_cap;
  const int base = int(tile) * kManifoldTile + int(threadIdx.x) * kManifoldItems;
  uint32_t cnt[kManifoldItems];
  uint32_t both = 0;  // manifolds, and their contacts (at most 4 x 2,048 in a tile) from bit 16 up
  int2 pr[kManifoldItems];
#pragma unroll
  for (int k = 0; k < kManifoldItems; ++k) {
    cnt[k] = base + k < npairs ? np.count[base + k] : 0u;
    pr[k] = base + k < npairs ? pairs[base + k] : int2{-1, -1};
    both += cnt[k] ? 1u + (cnt[k] << 16) : 0u;
  }
  uint32_t total;
  uint32_t m = block_exclusive(both, s_wave, total) & 0xffffu;
  if (threadIdx.x < 64) {
    const uint32_t before = scan_look_back(run, tile, total & 0xffffu);
    if (threadIdx.x == 0) {
      s_before = before;
      if (total) atomicAdd(&np.totals[0], total >> 16);
      if (tile == gridDim.x - 1) np.totals[1] = before + (total & 0xffffu);
    }
  }
  __syncthreads();
  m += s_before;
  int body = -1;  // body 1 of this lane's previous manifold
#pragma unroll
  for (int k = 0; k < kManifoldItems; ++k) {
    if (cnt[k] == 0u) continue;
    out.mbody[m] = pr[k];
    out.mfirst[m] = (base + k) * kPairSlots;
    out.mcount[m] = int(cnt[k]);
    // the body's first manifold: the smallest of what the lanes that hold some of its pairs offer
    if (out.bfirst && pr[k].x != body) atomicMin(reinterpret_cast<uint32_t*>(out.bfirst) + pr[k].x, m);
    body = pr[k].x;
    ++m;
  }
}

__global__ void __launch_bounds__(256) k_gather_contacts(DevContacts c, int M, const uint32_t* __restrict__ moff,
                                                        float4* dense, float4* dense_imp) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  const int first = c.mfirst[m], cnt = c.mcount[m];
  const long d0 = moff[m];
  for (int k = 0; k < cnt; ++k) {
    const float4* r = c.contact(first + k);
    float4* o = dense + (d0 + k) * kContactFields;
    for (int f = 0; f < kContactFields; ++f) o[f] = r[f];
    if (dense_imp) dense_imp[d0 + k] = c.imp[first + k];
  }
}

// The contacts as the arrays that a caller reads, four lanes per manifold, written straight to host memory
// (neighbouring lanes, neighbouring places). What bounds it is that link: 56 bytes a contact. Copying bodies and counts to the host
// for their prefix sum, that back, and the 48-byte records then took
// 328 us a call at 10,007 cuboids; this, with the copy out of the staging buffer, 87.
__global__ void __launch_bounds__(256) k_contacts_out(DevContacts c, int M, const uint32_t* __restrict__ moff, uint32_t cap,
                                                     ContactRows out, uint32_t* counted) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int m = t >> 2, k = t & 3;
  if (m >= M) return;
  const int cnt = c.mcount[m];
  if (m == M - 1 && k == 0) *counted = moff[m] + uint32_t(cnt);
  const uint32_t i = moff[m] + uint32_t(k);
  if (k >= cnt || i >= cap) return;
  const float4* r = c.contact(c.mfirst[m] + k);
  const float4 r0 = r[0], r1 = r[1], r2 = r[2];
  const int2 bb = c.mbody[m];
  if (out.row[0]) reinterpret_cast<int2*>(out.row[0])[i] = bb;
  if (out.row[1]) out.row[1][i] = r1.w;
  const float3 v[3] = {make_float3(r0.x, r0.y, r0.z), make_float3(r1.x, r1.y, r1.z), make_float3(r2.x, r2.y, r2.z)};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    if (!out.row[2 + a]) continue;
    float* o = out.row[2 + a] + 3 * long(i);
    o[0] = v[a].x;
    o[1] = v[a].y;
    o[2] = v[a].z;
  }
  if (out.row[5]) out.row[5][i] = r0.w;
}

}  // namespace

size_t manifold_tiles(int npairs) { return (size_t(npairs) + kManifoldTile - 1) / kManifoldTile; }

void launch_narrow_bins(const DevBodies& b, const int2* pairs, NarrowPhaseBufs& np, DevContacts out, hipStream_t s) {
  const int lanes = out.bfirst && out.bcount > np.pair_cap ? out.bcount : np.pair_cap;
  hipLaunchKernelGGL(k_np_bin, dim3(unsigned((lanes + 255) / 256)), dim3(256), 0, s, b, pairs, np, out);
}

// Grids for pair_cap pairs of either kind: what the lists hold is known on the device.
void launch_narrow_phase(const DevBodies& b, const int2* pairs, NarrowPhaseBufs& np, DevContacts out, hipStream_t s) {
  const unsigned P = unsigned(np.pair_cap);
  if (np.boxes)
    hipLaunchKernelGGL(k_np_boxes, dim3((P + kBoxBlock - 1) / kBoxBlock), dim3(kBoxBlock), 0, s, b, pairs, np, out);
  if (np.balls) hipLaunchKernelGGL(k_np_balls, dim3((P + 255) / 256), dim3(256), 0, s, b, pairs, np, out);
  const uint32_t tiles = uint32_t(manifold_tiles(np.pair_cap));
  hipLaunchKernelGGL(k_np_manifolds, dim3(tiles), dim3(kScanThreads), 0, s, pairs, np, out, np.scan->next(tiles, s));
}

void launch_gather_contacts(const DevContacts& c, int M, const uint32_t* moff, float4* dense,
                            float4* dense_imp, hipStream_t s) {
  if (M <= 0) return;
  hipLaunchKernelGGL(k_gather_contacts, dim3(unsigned((M + 255) / 256)), dim3(256), 0, s, c, M, moff, dense,
                     dense_imp);
}

void launch_contacts_out(const DevContacts& c, int M, const uint32_t* moff, uint32_t cap, const ContactRows& out,
                         uint32_t* counted, hipStream_t s) {
  hipLaunchKernelGGL(k_contacts_out, dim3(unsigned((4l * M + 255) / 256)), dim3(256), 0, s, c, M, moff, cap, out, counted);
}

}  // namespace nph
