// nphysics_amd/csrc/k_broadphase.hip -- broad phase: loose AABBs, search by boxes in Morton order, pair emission.
//
// Replaces ncollide's DBVTBroadPhase behind GeometricalWorld::perform_broad_phase
// (src/world/geometrical_world.rs:60, 285-312) and its DefaultCollisionFilter (:926-971):
//   * loose AABB rule (k_loose_update): tight = shape AABB at the collider position, merged with
//     the one at the predicted position when the CCD-phase sync sweeps the collider
//     (geometrical_world.rs:250-261, position0 -> position), loosened by margin + linear
//     prediction (collider.rs:542-549); the loose AABB is replaced by tight loosened by 0.01 only
//     when it no longer contains tight (the DBVT margin of geometrical_world.rs:60).
//   * pairs = every two bodies whose loose AABBs overlap (closed intervals), not the same body and
//     not both static; stored as (first, second) with first dynamic and second static or larger,
//     sorted.
// A world of one small scene is searched directly (k_direct). Others go by a tree 64 wide over the
// colliders in Morton order: boxes of 64 consecutive colliders and boxes of 64 of those (k_boxes, k_top),
// made anew at every search, while the order itself is sorted every kOrderAge-th time only: any order gives the same pairs,
// an old one slightly larger boxes. A wave
// searches for one body (k_search).
// Every body's partners go to its own fixed-capacity segment; a scan compacts the segments
// (k_compact). The result is deterministic and independent of thread timing. Algorithmic bytes: 124
// per body + 8 per pair. When only a few bodies' loose AABBs were replaced since the last search,
// the other bodies' segments are kept; the pair list is the same.
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "scan.hpp"
#include "stages.hpp"

namespace nph {

namespace {

__device__ __forceinline__ uint32_t f2ord(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// Replaces body i's loose AABB when it no longer contains `a` loosened by the query limit.
__device__ __forceinline__ bool loose_one(const DevBodies& b, int i, const aabb& a, aabb& loose) {
  const aabb tight = loosened(a, b.qlim[i]);
  if (contains(loose, tight)) return false;
  loose = loosened(tight, 0.01f);
  return true;
}

// One thread per body. passes: bit 0 the current pose of every body (of dynamic ones alone with
// bit 2 clear), bit 1 first the AABB swept from pos0/rot0 to the current pose (dynamic bodies; the
// CCD phase's sync, geometrical_world.rs:250-261). Both in one launch: a body's second pass reads
// nothing that another body's first one writes. changed[0..1]: the swept pass's counts, [2..3] the
// other's. Bodies replaced for the first time since the last pair build go to the dirty list.
__global__ void __launch_bounds__(256) k_loose_update(DevBodies b, int passes, uint32_t* changed, uint32_t* dirty,
                                                     int* list, uint32_t* list_count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const bool in = i < b.n;
  const bool dynamic = in && b.status[i] == STATUS_DYNAMIC;
  const bool work = in && (dynamic || (passes & 4));
  bool swept = false, final = false;
  if (work) {
    const int kind = b.shape[i];
    const f3 he = xyz(b.dims[i]);
    const q4 rot = toq(b.rot(i));
    const aabb a = shape_aabb(kind, he, xyz(b.pos(i)), rot);
    aabb loose{xyz(b.loose_mn[i]), xyz(b.loose_mx[i])};
    if ((passes & 2) && dynamic) {  // safe_position (rigid_body.rs:904-910): position0, with linear motion
                                    // interpolation the current rotation
      const q4 r0 = (b.ccd && (b.ccd[i] & 2)) ? rot : toq(b.rot0[i]);
      swept = loose_one(b, i, merged(shape_aabb(kind, he, xyz(b.pos0[i]), r0), a), loose);
    }
    if (passes & 1) final = loose_one(b, i, merged(a, a), loose);
    if (swept || final) {
      b.loose_mn[i] = f4(loose.mn, dynamic ? 1.0f : 0.0f);
      b.loose_mx[i] = f4(loose.mx, 0.0f);
    }
  }
  // counts and places in the dirty list, one atomic of each per workgroup: changed[0] every AABB the
  // swept pass replaced, [1] those of non-dynamic bodies, [2] and [3] the other pass's
  __shared__ uint32_t s_count[5][4];
  __shared__ uint32_t s_base;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool add = (swept || final) && dirty[i] == 0u;
  const uint64_t m[5] = {__ballot(swept), __ballot(swept && !dynamic), __ballot(final), __ballot(final && !dynamic),
                         __ballot(add)};
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < 5; ++k) s_count[k][wave] = uint32_t(__popcll(m[k]));
  }
  __syncthreads();
  if (threadIdx.x < 5) {
    const uint32_t c = s_count[threadIdx.x][0] + s_count[threadIdx.x][1] + s_count[threadIdx.x][2] + s_count[threadIdx.x][3];
    if (threadIdx.x == 4) s_base = c ? atomicAdd(list_count, c) : 0u;
    else if (c) atomicAdd(&changed[threadIdx.x], c);
  }
  __syncthreads();
  if (add) {
    uint32_t at = s_base + uint32_t(__popcll(m[4] & ((1ull << lane) - 1ull)));
    for (int w = 0; w < wave; ++w) at += s_count[4][w];
    dirty[i] = 1u;
    list[at] = i;
  }
}

__global__ void __launch_bounds__(256) k_bounds(DevBodies b, uint32_t* bounds) {
  __shared__ uint32_t s_b[6][256];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int t = threadIdx.x;
  uint32_t v[6] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0u, 0u, 0u};
  if (i < b.n) {
    const float4 mn = b.loose_mn[i], mx = b.loose_mx[i];
    const float cx = (mn.x + mx.x) * 0.5f, cy = (mn.y + mx.y) * 0.5f, cz = (mn.z + mx.z) * 0.5f;
    v[0] = v[3] = f2ord(cx);
    v[1] = v[4] = f2ord(cy);
    v[2] = v[5] = f2ord(cz);
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) s_b[k][t] = v[k];
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (t < off) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        s_b[k][t] = s_b[k][t] < s_b[k][t + off] ? s_b[k][t] : s_b[k][t + off];
        s_b[k + 3][t] = s_b[k + 3][t] > s_b[k + 3][t + off] ? s_b[k + 3][t] : s_b[k + 3][t + off];
      }
    }
    __syncthreads();
  }
  if (t < 3) atomicMin(&bounds[t], s_b[t][0]);
  else if (t < 6) atomicMax(&bounds[t], s_b[t][0]);
}

__device__ __forceinline__ uint32_t expand10(uint32_t v) {
  v &= 0x3ffu;
  v = (v | (v << 16)) & 0x030000ffu;
  v = (v | (v << 8)) & 0x0300f00fu;
  v = (v | (v << 4)) & 0x030c30c3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

// Coordinate quantised to `levels` (2^bits - 1) steps of the centroid bounds.
__device__ __forceinline__ uint32_t quant(float c, float lo, float hi, float levels, uint32_t top) {
  const float ext = hi - lo;
  float u = ext > 0.0f ? (c - lo) / ext : 0.5f;
  u = u < 0.0f ? 0.0f : (u > 1.0f ? 1.0f : u);
  const uint32_t q = uint32_t(u * levels);
  return q > top ? top : q;
}

// Key = scene << 3m | Morton code of the loose-AABB centroid with m bits per axis,
// m = (30 - scene_bits) / 3 (10 for a single scene).
__global__ void __launch_bounds__(256) k_morton(DevBodies b, const uint32_t* bounds, int scene_bits,
                                               uint32_t* keys, uint32_t* vals) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= b.n) return;
  const int m = (30 - scene_bits) / 3;
  const uint32_t top = (1u << m) - 1u;
  const float levels = float(top);
  const float lx = ord2f(bounds[0]), ly = ord2f(bounds[1]), lz = ord2f(bounds[2]);
  const float hx = ord2f(bounds[3]), hy = ord2f(bounds[4]), hz = ord2f(bounds[5]);
  const float4 mn = b.loose_mn[i], mx = b.loose_mx[i];
  const float cx = (mn.x + mx.x) * 0.5f, cy = (mn.y + mx.y) * 0.5f, cz = (mn.z + mx.z) * 0.5f;
  const uint32_t x = quant(cx, lx, hx, levels, top), y = quant(cy, ly, hy, levels, top),
                 z = quant(cz, lz, hz, levels, top);
  const uint32_t morton = (expand10(x) << 2) | (expand10(y) << 1) | expand10(z);
  keys[i] = scene_bits ? (uint32_t(b.scene[i]) << (3 * m)) | morton : morton;
  vals[i] = uint32_t(i);
}

// Box of 64 consecutive colliders of the order, or of 64 such boxes: bounds, the scenes of its
// colliders and the largest index a partner can have in it (no limit with a non-dynamic collider).
__device__ __forceinline__ void wave_box(aabb& a, int& smin, int& smax, int& top) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    a.mn.x = fminf(a.mn.x, __shfl_xor(a.mn.x, off));
    a.mn.y = fminf(a.mn.y, __shfl_xor(a.mn.y, off));
    a.mn.z = fminf(a.mn.z, __shfl_xor(a.mn.z, off));
    a.mx.x = fmaxf(a.mx.x, __shfl_xor(a.mx.x, off));
    a.mx.y = fmaxf(a.mx.y, __shfl_xor(a.mx.y, off));
    a.mx.z = fmaxf(a.mx.z, __shfl_xor(a.mx.z, off));
    smin = min(smin, __shfl_xor(smin, off));
    smax = max(smax, __shfl_xor(smax, off));
    top = max(top, __shfl_xor(top, off));
  }
}

constexpr float kInf = __builtin_huge_valf();
constexpr int kDynBit = 1 << 30;

// One wave per box: the colliders' loose AABBs in the order (mn.w: index and dynamic flag, mx.w: scene)
// and their box.
__global__ void __launch_bounds__(256) k_boxes(DevBodies b, BroadPhaseBufs bp) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63;
  const bool in = p < b.n;
  if ((p & ~63) >= b.n) return;
  aabb a{{kInf, kInf, kInf}, {-kInf, -kInf, -kInf}};
  int smin = 0x7fffffff, smax = -1, top = -1;
  if (in) {
    const int o = int(bp.vals[p]);
    const float4 mn = b.loose_mn[o], mx = b.loose_mx[o];
    const bool dyn = mn.w != 0.0f;
    const int sc = b.scene[o];
    bp.leaf_mn[p] = f4(xyz(mn), __int_as_float(o | (dyn ? kDynBit : 0)));
    bp.leaf_mx[p] = f4(xyz(mx), __int_as_float(sc));
    a = aabb{xyz(mn), xyz(mx)};
    smin = smax = sc;
    top = dyn ? o : 0x7fffffff;
  }
  wave_box(a, smin, smax, top);
  if (lane == 0) {
    bp.box_mn[p >> 6] = f4(a.mn, __int_as_float(smin));
    bp.box_mx[p >> 6] = f4(a.mx, __int_as_float(smax));
    bp.box_top[p >> 6] = top;
  }
}

// One wave per box of boxes, stored after the nbox boxes.
__global__ void __launch_bounds__(64) k_top(BroadPhaseBufs bp, int nbox) {
  const int k = blockIdx.x * 64 + threadIdx.x;
  aabb a{{kInf, kInf, kInf}, {-kInf, -kInf, -kInf}};
  int smin = 0x7fffffff, smax = -1, top = -1;
  if (k < nbox) {
    const float4 mn = bp.box_mn[k], mx = bp.box_mx[k];
    a = aabb{xyz(mn), xyz(mx)};
    smin = __float_as_int(mn.w);
    smax = __float_as_int(mx.w);
    top = bp.box_top[k];
  }
  wave_box(a, smin, smax, top);
  if (threadIdx.x == 0) {
    bp.box_mn[nbox + blockIdx.x] = f4(a.mn, __int_as_float(smin));
    bp.box_mx[nbox + blockIdx.x] = f4(a.mx, __int_as_float(smax));
    bp.box_top[nbox + blockIdx.x] = top;
  }
}

// All six comparisons evaluated (with && it would stop at the first that fails: a branch each).
__device__ __forceinline__ bool overlap(const aabb& a, const aabb& c) {
  return (a.mn.x <= c.mx.x) & (c.mn.x <= a.mx.x) & (a.mn.y <= c.mx.y) & (c.mn.y <= a.mx.y) & (a.mn.z <= c.mx.z) &
         (c.mn.z <= a.mx.z);
}

// Whether the segments of bodies that nothing happened to are kept: the counts of this step's
// loose-AABB passes are on the device, so no readback stands between the passes and the search.
__device__ __forceinline__ bool search_incremental(const BroadPhaseBufs& bp, const SearchRun& r, int n) {
  const uint32_t all = bp.changed[0] + bp.changed[2], fixed = bp.changed[1] + bp.changed[3];
  return r.may_increment && fixed == 0u && all <= uint32_t(kept_limit(n));
}

// ---- search by boxes -----------------------------------------------------------------------------
// A wave searches for one body, its bounds in scalar registers: it tests 64 upper boxes at a time, then the 64 boxes
// of each that overlaps, then the 64 colliders of each of those (its lanes the boxes or colliders), and a ballot tells each
// hit its place in the segment. The loads of the next box are in flight while one is tested. A body meets three to
// five boxes, so about eight tests of some forty instructions, however many colliders there are. (One wave for the 64
// bodies of a box, descending by their common bounds, has fewer tests but the slowest wave of a launch, one whose
// bodies straddle a jump of the Morton curve, held it up: 370 us at 8,001 bodies and 1.75 ms at 99,996.)
// Measured: 14 us at 8,001 bodies, 29 us at 21,004 and 121 us at 99,996 in piles. With k_boxes, k_top and the
// compaction the whole phase takes 58, 76 and 190 us there; the binary tree it replaces (topology, atomic
// refit, packing and a stack per lane, on a sort at every build) took 268, 337 and 526 us.
//
// Incremental form: a body searches anew if its loose AABB was replaced (dirty), if it held a dirty
// partner, or if a dirty body with a larger index now overlaps it; the others keep their segments.
template <bool kScenes>
__global__ void __launch_bounds__(256) k_search(DevBodies b, BroadPhaseBufs bp, SearchRun r) {
  const int lane = threadIdx.x & 63, n = b.n;
  const uint64_t below = (1ull << lane) - 1ull;
  const int p = __builtin_amdgcn_readfirstlane(int((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
  if (p >= n) return;
  const float4 mn = bp.leaf_mn[p], mx = bp.leaf_mx[p];
  const int code = __float_as_int(mn.w), q = code & (kDynBit - 1), sc = __float_as_int(mx.w);
  if ((code & kDynBit) == 0) {
    if (lane == 0) bp.cand_count[q] = 0u;
    return;
  }
  const aabb Q{xyz(mn), xyz(mx)};
  const uint4 qg = b.groups ? b.groups[q] : uint4{};
  int* seg = bp.cand + long(q) * r.cap;
  auto partner = [&](int o, bool dyn, int osc, const aabb& B) {
    bool hit = overlap(Q, B) & (o != q) & (!dyn | (o > q));
    if (kScenes) hit = hit & (osc == sc);
    if (b.groups) hit = hit && groups_interact(qg, b.groups[o]);
    return hit;
  };
  if (search_incremental(bp, r, n) && bp.dirty[q] == 0u) {
    bool again = false;
    const int c = min(int(bp.cand_count[q]), r.cap), nd = int(*bp.list_count);
    for (int k = lane; k < c; k += 64) again = again || bp.dirty[seg[k]] != 0u;
    for (int k = lane; k < nd; k += 64) {  // the dirty bodies are all dynamic here
      const int o = bp.list[k];
      again = again || partner(o, true, kScenes ? b.scene[o] : 0, aabb{xyz(b.loose_mn[o]), xyz(b.loose_mx[o])});
    }
    if (!__any(again)) return;
  }
  auto enter = [&](int k) {
    const float4 cmn = bp.box_mn[k], cmx = bp.box_mx[k];
    bool ok = overlap(Q, aabb{xyz(cmn), xyz(cmx)}) & (bp.box_top[k] > q);
    if (kScenes) ok = ok & (__float_as_int(cmn.w) <= sc) & (__float_as_int(cmx.w) >= sc);
    return ok;
  };
  uint32_t cnt = 0;
  const int nbox = (n + 63) >> 6, ntop = (nbox + 63) >> 6;
  for (int t0 = 0; t0 < ntop; t0 += 64) {
    uint64_t mt = 1ull;
    if (ntop > 1) {
      const int t = t0 + lane;
      mt = __ballot((t < ntop) & enter(nbox + (t < ntop ? t : t0)));
    }
    while (mt) {
      const int t = t0 + __ffsll(static_cast<long long>(mt)) - 1;
      mt &= mt - 1;
      const int c = t * 64 + lane;
      uint64_t mb = __ballot((c < nbox) & enter(c < nbox ? c : nbox - 1));
      float4 nmn{}, nmx{};
      auto load = [&](int box) {
        const int k = box * 64 + lane < n ? box * 64 + lane : n - 1;
        nmn = bp.leaf_mn[k];
        nmx = bp.leaf_mx[k];
      };
      int next = mb ? t * 64 + __ffsll(static_cast<long long>(mb)) - 1 : -1;
      if (next >= 0) load(next);
      while (next >= 0) {
        const int box = next;
        const float4 omn = nmn, omx = nmx;
        mb &= mb - 1;
        next = mb ? t * 64 + __ffsll(static_cast<long long>(mb)) - 1 : -1;
        if (next >= 0) load(next);
        const int ocode = __float_as_int(omn.w), o = ocode & (kDynBit - 1);
        const bool hit = (box * 64 + lane < n) & partner(o, (ocode & kDynBit) != 0, __float_as_int(omx.w),
                                                        aabb{xyz(omn), xyz(omx)});
        const uint64_t m = __ballot(hit);
        const uint32_t at = cnt + uint32_t(__popcll(m & below));
        if (hit && at < uint32_t(r.cap)) seg[at] = o;
        cnt += uint32_t(__popcll(m));
      }
    }
  }
  if (lane == 0) {
    bp.cand_count[q] = cnt;
    if (cnt > uint32_t(r.cap)) atomicMax(&bp.stats[0], cnt);
  }
}

// ---- direct pair search ------------------------------------------------------------------------
// A world of one scene with at most kDirectBodies colliders: a wave takes kDirectGroup bodies and tests
// them against all colliders, 64 at a time in ascending order, and a ballot per body and 64 tells
// each hit its place, so that the segments come out sorted. There the time is the few launches and
// the loads' latency (kDirectAhead of them in flight), which boxes would only add to; above, the
// tests do, growing with the square: 13 us at 1,001 bodies, where the boxes and their search take 12 us
// and ordering and sorting as much again, and 98 us at 8,001, where they take 22 us.
constexpr int kDirectGroup = 4;
constexpr int kDirectAhead = 4;

__global__ void __launch_bounds__(256) k_direct(DevBodies b, BroadPhaseBufs bp, SearchRun r) {
  constexpr int G = kDirectGroup;
  const int lane = threadIdx.x & 63, n = b.n;
  const uint64_t below = (1ull << lane) - 1ull;
  const int first = __builtin_amdgcn_readfirstlane(int((blockIdx.x * blockDim.x + threadIdx.x) >> 6)) * G;
  if (first >= n) return;
  int q[G];
  uint32_t cnt[G];
  bool todo[G];
  aabb Q[G];
  uint4 qg[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    cnt[g] = 0;
    q[g] = first + g < n ? first + g : n - 1;
    const float4 mn = b.loose_mn[q[g]], mx = b.loose_mx[q[g]];
    todo[g] = first + g < n && mn.w != 0.0f;  // dynamic
    if (first + g < n && !todo[g] && lane == 0) bp.cand_count[q[g]] = 0;
    Q[g] = aabb{xyz(mn), xyz(mx)};
    qg[g] = b.groups ? b.groups[q[g]] : uint4{};
  }
  auto hits = [&](int g, int o, bool dyn, const aabb& B) {
    const bool hit = overlap(Q[g], B) & (o != q[g]) & (!dyn | (o > q[g]));
    return b.groups ? hit && groups_interact(qg[g], b.groups[o]) : hit;
  };
  if (search_incremental(bp, r, n)) {
    const int nd = int(*bp.list_count);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (!todo[g] || bp.dirty[q[g]] != 0u) continue;
      bool again = false;
      const int c = min(int(bp.cand_count[q[g]]), r.cap);
      for (int k = lane; k < c; k += 64) again = again || bp.dirty[bp.cand[long(q[g]) * r.cap + k]] != 0u;
      for (int k = lane; k < nd; k += 64) {  // the dirty bodies are all dynamic here
        const int o = bp.list[k];
        again = again || hits(g, o, true, aabb{xyz(b.loose_mn[o]), xyz(b.loose_mx[o])});
      }
      todo[g] = __any(again);
    }
  }
  if (!(todo[0] || todo[1] || todo[2] || todo[3])) return;
  // colliders [0, fixed_end) hold the last non-dynamic one; the dynamic ones before the first body have
  // smaller indices
  for (int c = 0; c < n; c += 64 * kDirectAhead) {
    if (c >= r.fixed_end && c + 63 < first) c = first & ~63;
    float4 mn[kDirectAhead], mx[kDirectAhead];
#pragma unroll
    for (int u = 0; u < kDirectAhead; ++u) {
      const int o = c + 64 * u + lane;
      mn[u] = b.loose_mn[o < n ? o : n - 1];
      mx[u] = b.loose_mx[o < n ? o : n - 1];
    }
#pragma unroll
    for (int u = 0; u < kDirectAhead; ++u) {
      if (c + 64 * u >= n) break;
      const int o = c + 64 * u + lane;
      const bool dyn = mn[u].w != 0.0f;
      const aabb B{xyz(mn[u]), xyz(mx[u])};
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if (!todo[g]) continue;
        const bool hit = (o < n) & hits(g, o < n ? o : n - 1, dyn, B);
        const uint64_t m = __ballot(hit);
        if (!m) continue;
        const uint32_t k = cnt[g] + uint32_t(__popcll(m & below));
        if (hit && k < uint32_t(r.cap)) bp.cand[long(q[g]) * r.cap + k] = o;
        cnt[g] += uint32_t(__popcll(m));
      }
    }
  }
  if (lane == 0) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (!todo[g]) continue;
      bp.cand_count[q[g]] = cnt[g];
      if (cnt[g] > uint32_t(r.cap)) atomicMax(&bp.stats[0], cnt[g]);
    }
  }
}

// ---- compaction ----------------------------------------------------------------------------------
// The segments, one after another in body order, into the pair list, and every pair into the narrow
// phase's list of its kind. One launch: a tile of kCompactBodies bodies looks back for the pairs
// before it (scan.hpp). The pairs of a tile are written by consecutive lanes, each finding its body
// in the tile's prefix sums in LDS (one lane per body wrote 8-byte pieces and waited for its own
// reads: 52 us at 100,000 bodies beside the offsets' four launches; now 11 us at
// 1,001 bodies and 38 us at 99,996). With kSort the
// segments are in any order, and a pair's place is the number of smaller partners in its segment
// (the direct search leaves them sorted). It also clears what
// the next loose-AABB pass and this step's narrow phase start from: the dirty flags and the manifold
// index. No pair at or above pair_cap is written: the caller sees the count and runs it again.
constexpr int kCompactBodies = 256;

template <bool kSort>
__global__ void __launch_bounds__(kScanThreads) k_compact(DevBodies b, BroadPhaseBufs bp, int cap, ScanRun run,
                                                          PairOut o) {
  __shared__ uint32_t s_wave[kScanWaves];
  __shared__ uint32_t s_tile, s_before, s_box, s_ball;
  __shared__ uint32_t s_off[kCompactBodies];
  const uint32_t tile = scan_tile(run, &s_tile);
  if (tile >= gridDim.x) return;  // only after a launch that failed: its tickets were never taken
  const int t = threadIdx.x;
  const int q = int(tile) * kCompactBodies + t;
  uint32_t c = 0;
  if (q < b.n) {
    c = bp.cand_count[q];
    c = c < uint32_t(cap) ? c : uint32_t(cap);
    bp.dirty[q] = 0u;
    if (o.bfirst) o.bfirst[q] = -1;
  }
  uint32_t total;
  s_off[t] = block_exclusive(c, s_wave, total);
  if (t < 64) {
    const uint32_t before = scan_look_back(run, tile, total);
    if (t == 0) {
      s_before = before;
      if (tile == gridDim.x - 1) *o.npairs = before + total;
    }
  }
  __syncthreads();
  const uint32_t before = s_before;
  // kGo pairs per lane in one go, so that the places in the two lists take one atomic of each per go
  constexpr int kGo = 8;
  for (uint32_t k0 = 0; k0 < total; k0 += kGo * kScanThreads) {
    uint32_t at[kGo];
    bool live[kGo], box[kGo];
    uint32_t boxes = 0, balls = 0;
#pragma unroll
    for (int u = 0; u < kGo; ++u) {
      const uint32_t k = k0 + uint32_t(u * kScanThreads + t);
      live[u] = box[u] = false;
      if (k >= total) continue;
      int lo = 0, hi = kCompactBodies - 1;  // the last body whose offset is <= k: it has pairs
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s_off[mid] <= k) lo = mid;
        else hi = mid - 1;
      }
      const int x = int(tile) * kCompactBodies + lo;
      const int* seg = bp.cand + long(x) * cap;
      const int y = seg[k - s_off[lo]];
      at[u] = before + k;
      if (kSort) {
        const uint32_t c = (lo + 1 < kCompactBodies ? s_off[lo + 1] : total) - s_off[lo];
        at[u] = before + s_off[lo];
        for (uint32_t j = 0; j < c; ++j) at[u] += seg[j] < y ? 1u : 0u;
      }
      if (at[u] >= uint32_t(o.pair_cap)) continue;
      bp.pairs[at[u]] = make_int2(x, y);
      live[u] = true;
      box[u] = b.shape[x] == SHAPE_CUBOID && b.shape[y] == SHAPE_CUBOID;
      if (box[u]) ++boxes;
      else ++balls;
    }
    uint32_t nbox, nball;
    uint32_t ab = block_exclusive(boxes, s_wave, nbox);
    uint32_t aa = block_exclusive(balls, s_wave, nball);
    if (t == 0 && nbox) s_box = atomicAdd(o.nbox, nbox);
    if (t == 64 && nball) s_ball = atomicAdd(o.nball, nball);
    __syncthreads();
    ab += s_box;
    aa += s_ball;
#pragma unroll
    for (int u = 0; u < kGo; ++u) {
      if (!live[u]) continue;
      if (box[u]) o.perm[ab++] = at[u];
      else o.perm[uint32_t(o.pair_cap) - 1u - aa++] = at[u];
    }
    __syncthreads();
  }
}

inline unsigned nb(long n) { return unsigned((n + 255) / 256); }

}  // namespace

void launch_loose_update(const DevBodies& b, int passes, BroadPhaseBufs& bp, hipStream_t s) {
  if (b.n == 0) return;
  hipLaunchKernelGGL(k_loose_update, dim3(nb(b.n)), dim3(256), 0, s, b, passes, bp.changed, bp.dirty, bp.list,
                     bp.list_count);
}

void launch_order(const DevBodies& b, BroadPhaseBufs& bp, hipStream_t s) {
  const int n = b.n;
  if (n == 0) return;
  fill_u32(bp.bounds, 0xffffffffu, 3, s);
  fill_u32(bp.bounds + 3, 0u, 3, s);
  hipLaunchKernelGGL(k_bounds, dim3(nb(n)), dim3(256), 0, s, b, bp.bounds);
  hipLaunchKernelGGL(k_morton, dim3(nb(n)), dim3(256), 0, s, b, bp.bounds, bp.scene_bits, bp.keys, bp.vals);
  radix_sort_pairs(bp.keys, bp.vals, bp.keys_alt, bp.vals_alt, n, 30, bp.tmp, *bp.scan, s);
}

void launch_search(const DevBodies& b, BroadPhaseBufs& bp, const SearchRun& r, hipStream_t s) {
  const int n = b.n;
  if (n == 0) return;
  if (r.direct) {
    // four waves per workgroup
    hipLaunchKernelGGL(k_direct, dim3(unsigned((n + 4 * kDirectGroup - 1) / (4 * kDirectGroup))), dim3(256), 0, s, b, bp, r);
    return;
  }
  const int nbox = (n + 63) / 64, ntop = (nbox + 63) / 64;
  hipLaunchKernelGGL(k_boxes, dim3(nb(n)), dim3(256), 0, s, b, bp);
  if (ntop > 1) hipLaunchKernelGGL(k_top, dim3(unsigned(ntop)), dim3(64), 0, s, bp, nbox);
  const dim3 grid(unsigned((n + 3) / 4));  // four waves per workgroup
  if (bp.scene_bits) hipLaunchKernelGGL(k_search<true>, grid, dim3(256), 0, s, b, bp, r);
  else hipLaunchKernelGGL(k_search<false>, grid, dim3(256), 0, s, b, bp, r);
}

size_t compact_tiles(int n) { return (size_t(n) + kCompactBodies - 1) / kCompactBodies; }

void launch_compact_pairs(const DevBodies& b, BroadPhaseBufs& bp, int cap, bool sorted, const PairOut& o, hipStream_t s) {
  if (b.n == 0) return;
  const uint32_t tiles = uint32_t(compact_tiles(b.n));
  const ScanRun run = bp.scan->next(tiles, s);
  if (sorted) hipLaunchKernelGGL(k_compact<false>, dim3(tiles), dim3(kScanThreads), 0, s, b, bp, cap, run, o);
  else hipLaunchKernelGGL(k_compact<true>, dim3(tiles), dim3(kScanThreads), 0, s, b, bp, cap, run, o);
}

}  // namespace nph
