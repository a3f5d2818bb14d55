// nphysics_amd/csrc/k_ccd.hip -- continuous collision detection: times of impact, the impact
// queue, and the substep island.
//
// Restates MechanicalWorld::predict_next_impacts and the island traversal of solve_ccd
// (src/world/mechanical_world.rs:400-557, 630-861) with TOIEntry::try_from_colliders (:946-1022):
//   * k_ccd_first_pass: every broad-phase pair with a CCD-enabled side gets a CCD slot and its time
//     of impact up to the step's end (conservative advancement, np_geometry.hpp); impacts within
//     the window become the slots' keys, later ones lower the earliest-later time;
//   * k_ccd_events, one workgroup, takes the earliest impact (ties by pair index) again and again,
//     confirms pairs of two frozen bodies only at the later freeze time, and freezes the two bodies
//     (their keys: a static collider shares its static body's); then the CCD slots of the frozen
//     bodies' dynamic colliders are re-swept with the frozen bodies held at their freeze poses;
//   * k_ccd_foresee, on the whole chip, does those re-sweeps beforehand: a body not frozen yet will freeze
//     at its earliest key unless an event before changes that, so the times of impact of its slots
//     with it held there are recorded with the freeze time they hold for. An event takes the
//     recorded times where the freeze time is the one that came true and computes the others itself; after
//     kEventMisses events with such others it stops for k_ccd_foresee to look again from there;
//   * the island of a substep grows in rounds: the dynamic bodies of every pair touching a
//     traversed collider are moved to their impact time (k_ccd_touch, k_ccd_prepare; the dynamics
//     update of the substep, no gravity, forces cleared), those pairs' manifolds are computed by
//     the narrow phase at the moved poses, and the dynamic bodies of the non-empty ones are
//     traversed from the next round (k_ccd_grow, k_ccd_merge);
//   * k_ccd_validate (validate_advancement of the impacting bodies) and k_ccd_clamp (bodies still
//     predicted to impact go back to the start of their motion, rigid_body.rs:530-537).
// The queue is serial by nature; what an event does is a few hundred instructions, while the
// time-of-impact queries (the arithmetic) have sixteen lanes each, over all compute units.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "np_geometry.hpp"
#include "stages.hpp"

namespace nph {

namespace {

constexpr int kEventBlock = 512;
// Events with times not foreseen, some 10 us each, before the next round (2 to 16: within 2% of each other).
constexpr int kEventMisses = 4;

__device__ __forceinline__ unsigned long long toi_key(float toi, int pair) {
  return (static_cast<unsigned long long>(__float_as_uint(toi)) << 32) | static_cast<unsigned long long>(uint32_t(pair));
}
__device__ __forceinline__ float key_toi(unsigned long long k) { return __uint_as_float(uint32_t(k >> 32)); }
__device__ __forceinline__ int key_pair(unsigned long long k) { return int(uint32_t(k & 0xffffffffull)); }

// Body::part_motion (rigid_body.rs:539-553): static bodies at their pose; with linear motion
// interpolation from (position0, current rotation); else from position0 with rotation.
__device__ __forceinline__ CcdMotion part_motion(const DevBodies& b, int i, float t0) {
  CcdMotion m;
  m.t0 = t0;
  m.v = xyz(b.linvel[i]);
  m.w = xyz(b.angvel[i]);
  if (b.status[i] != STATUS_DYNAMIC) {
    m.kind = MOTION_STATIC;
    m.t0p = xyz(b.pos(i));
    m.q0 = toq(b.rot(i));
  } else if (b.ccd[i] & 2) {
    m.kind = MOTION_LINEAR;
    m.t0p = xyz(b.pos0[i]);
    m.q0 = toq(b.rot(i));
  } else {
    m.kind = MOTION_ROTATING;
    m.t0p = xyz(b.pos0[i]);
    m.q0 = toq(b.rot0[i]);
  }
  return m;
}

// ---- time of impact on sixteen lanes ----
// Sixteen lanes (one DPP row) share a query, all with the same arguments: lanes 0-7 move body 1 and lanes 8-15 body 2, each
// lane measures one of the 15 axes of the cuboid / cuboid separation, and the largest is found by
// four permutation steps. The expressions of the scalar form (of toi_separation for the axes), in its order, so the
// same bits; a single lane takes some 1,000 instructions per iterate, these some 350.
constexpr int kToiLanes = 16;

template <int Ctrl>
__device__ __forceinline__ float row_perm(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), Ctrl, 0xf, 0xf, true));
}
template <int Ctrl>
__device__ __forceinline__ void max_axis_step(float& s, int& r) {
  const float os = row_perm<Ctrl>(s);
  const int orr = __builtin_amdgcn_mov_dpp(r, Ctrl, 0xf, 0xf, true);
  const bool other = os > s || (os == s && orr < r);
  s = other ? os : s;
  r = other ? orr : r;
}
constexpr int kQuadXor1 = 0xb1, kQuadXor2 = 0x4e, kHalfMirror = 0x141, kMirror = 0x140;

// toi_separation of two cuboids whose axes are the columns of RA and RB; r: the lane's place in its row.
__device__ __forceinline__ float boxes_separation(f3 h1, const m33& RA, f3 h2, const m33& RB, f3 d, int r, f3& n) {
  f3 a[3], b[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    a[i] = mcol(RA, i);
    b[i] = mcol(RB, i);
  }
  // lanes 0-2: the faces of A, 3-5: of B, 6-14: the edge axes, in toi_separation's order
  const int e = r < 6 ? 0 : r - 6;
  const int i = r < 3 ? r : (r < 6 ? 0 : (e * 11) >> 5);  // e / 3 for e < 10
  const int j = r < 6 ? (r < 3 ? 0 : r - 3) : e - 3 * i;
  const f3 ai = pick(i == 0, a[0], pick(i == 1, a[1], a[2])), bj = pick(j == 0, b[0], pick(j == 1, b[1], b[2]));
  const f3 c = cross(ai, bj);
  const f3 L = pick(r < 3, ai, pick(r < 6, bj, c));
  float l = 1.0f, s = -INFINITY;
  const float l2 = dot(c, c);
  if (r >= 6) l = sqrtf(l2);
  const float pa = (h1.x * fabsf(dot(a[0], L)) + h1.y * fabsf(dot(a[1], L))) + h1.z * fabsf(dot(a[2], L));
  const float pb = (h2.x * fabsf(dot(b[0], L)) + h2.y * fabsf(dot(b[1], L))) + h2.z * fabsf(dot(b[2], L));
  const float ra = r < 3 ? comp(h1, i) : pa, rb = (r >= 3 && r < 6) ? comp(h2, j) : pb;
  if (r < 6 || (r < 15 && !(l2 < 1e-6f))) {
    const float m = (fabsf(dot(d, L)) - (ra + rb)) / l;
    s = m > s ? m : s;  // never a NaN
  }
  int best = r;
  max_axis_step<kQuadXor1>(s, best);
  max_axis_step<kQuadXor2>(s, best);
  max_axis_step<kHalfMirror>(s, best);
  max_axis_step<kMirror>(s, best);
  f3 axis{__shfl(L.x, best, kToiLanes), __shfl(L.y, best, kToiLanes), __shfl(L.z, best, kToiLanes)};
  const float scale = __shfl(l, best, kToiLanes);
  if (scale != 1.0f) axis = f3{axis.x / scale, axis.y / scale, axis.z / scale};
  n = dot(d, axis) < 0.0f ? neg(axis) : axis;
  return s;
}

// TOIEntry::try_from_colliders for bodies i, j with freeze times f1, f2 (< 0: not frozen): the
// global time of impact up to end_time.
__device__ bool pair_toi(const DevBodies& b, const CcdBufs& c, int i, int j, float f1, float f2, float end_time,
                         float target, int on_penetration, int r, float* out) {
  const bool second = r >= kToiLanes / 2;
  const float bt1 = c.body_time[i], bt2 = c.body_time[j];
  const float time1 = f1 >= 0.0f ? f1 : bt1;
  const float time2 = f2 >= 0.0f ? f2 : bt2;
  const float start = time1 > time2 ? time1 : time2;
  const float o = (second ? time2 : time1) - start;
  const float f = second ? f2 : f1;
  CcdMotion m = part_motion(b, second ? j : i, o);
  if (f >= 0.0f) {
    m.at((f + o) - (second ? bt2 : bt1), m.t0p, m.q0);
    m.kind = MOTION_STATIC;
  }
  const int k1 = b.shape[i], k2 = b.shape[j];
  const f3 h1 = xyz(b.dims[i]), h2 = xyz(b.dims[j]);
  const float max_toi = end_time - start;
  // what turns and moves: both bodies' velocities in every lane
  const f3 z{0.0f, 0.0f, 0.0f};
  const f3 v = m.kind == MOTION_STATIC ? z : m.v;
  const f3 w = m.kind == MOTION_ROTATING ? m.w : z;
  const float reach = sqrtf(dot(w, w)) * (second ? rotation_reach(k2, h2) : rotation_reach(k1, h1));
  const float reach_o = row_perm<kMirror>(reach);
  const float spin = second ? reach_o + reach : reach + reach_o;
  const f3 vo{row_perm<kMirror>(v.x), row_perm<kMirror>(v.y), row_perm<kMirror>(v.z)};
  const f3 dv = second ? sub(v, vo) : sub(vo, v);
  float tau = 0.0f;
  int status = TOI_OUT_OF_ITERATIONS;
  for (int it = 0; it < kToiMaxIterations; ++it) {
    f3 p, n;
    q4 q;
    m.at(tau, p, q);
    const f3 po{row_perm<kMirror>(p.x), row_perm<kMirror>(p.y), row_perm<kMirror>(p.z)};
    const f3 p1 = pick(second, po, p), p2 = pick(second, p, po);
    float d;
    if (k1 == SHAPE_BALL || k2 == SHAPE_BALL) {
      const q4 qo{row_perm<kMirror>(q.i), row_perm<kMirror>(q.j), row_perm<kMirror>(q.k), row_perm<kMirror>(q.w)};
      d = toi_separation(k1, h1, p1, second ? qo : q, k2, h2, p2, second ? q : qo, n);
    } else {
      const m33 R = qmat(q);
      m33 R1, R2;
#pragma unroll
      for (int x = 0; x < 3; ++x)
#pragma unroll
        for (int y = 0; y < 3; ++y) {
          const float ro = row_perm<kMirror>(R.m[x][y]);
          R1.m[x][y] = second ? ro : R.m[x][y];
          R2.m[x][y] = second ? R.m[x][y] : ro;
        }
      d = boxes_separation(h1, R1, h2, R2, sub(p2, p1), r, n);
    }
    if (it == 0 && d < 0.0f) {
      status = TOI_PENETRATING;
      break;
    }
    if (d <= target + kToiTolerance) {
      status = TOI_CONVERGED;
      break;
    }
    const float a = spin - dot(dv, n);
    if (!(a > 0.0f)) return false;
    tau = tau + (d - target) / a;
    if (tau > max_toi) return false;
  }
  if (!on_penetration && status == TOI_PENETRATING) return false;
  *out = start + tau;
  return true;
}

__global__ void __launch_bounds__(256) k_ccd_begin(int n, CcdBufs c) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kCcdWords) c.ctl[i] = i == kCcdMinAfter ? 0x7f800000u : 0u;  // +inf
  if (i >= n) return;
  c.frozen[i] = -1.0f;
  c.deg[i] = 0u;
  c.fill[i] = 0u;
}

constexpr unsigned long long kNoKey = ~0ull;
constexpr int kFirstPairs = 64;  // pairs of one workgroup of the first pass

// Wave 0 gives the CCD pairs of the workgroup's 64 their slots, then its sixteen rows of lanes take those in turn.
__global__ void __launch_bounds__(256) k_ccd_first_pass(DevBodies b, const int2* __restrict__ pairs, int npairs,
                                                        CcdBufs c, float end_time, float dt0, float target,
                                                        int on_penetration) {
  __shared__ int s_pair[kFirstPairs];
  __shared__ int2 s_body[kFirstPairs];
  __shared__ uint32_t s_first;
  __shared__ int s_n;
  const int t = threadIdx.x;
  if (t < 64) {
    const int p = blockIdx.x * kFirstPairs + t;
    const int2 pr = p < npairs ? pairs[p] : int2{0, 0};
    const bool on = p < npairs && ((b.ccd[pr.x] | b.ccd[pr.y]) & 1);
    const unsigned long long m = __ballot(on);
    const int at = __popcll(m & ((1ull << t) - 1ull));
    uint32_t first = 0;
    if (t == 0) {
      if (m) first = atomicAdd(&c.ctl[kCcdSlots], uint32_t(__popcll(m)));
      s_first = first;
      s_n = __popcll(m);
    }
    first = uint32_t(__builtin_amdgcn_readfirstlane(int(first)));
    if (on) {
      s_pair[at] = p;
      s_body[at] = pr;
      const uint32_t slot = first + uint32_t(at);
      const bool st1 = b.status[pr.x] != STATUS_DYNAMIC, st2 = b.status[pr.y] != STATUS_DYNAMIC;
      c.slot_pair[slot] = p;
      c.slot_bodies[slot] =
          int4{pr.x, pr.y, b.ccd_key[pr.x] | (st1 ? kSlotStatic : 0), b.ccd_key[pr.y] | (st2 ? kSlotStatic : 0)};
      c.seen_at[2 * slot] = c.seen_at[2 * slot + 1] = -1.0f;
      if (!st1) atomicAdd(&c.deg[pr.x], 1u);
      if (!st2) atomicAdd(&c.deg[pr.y], 1u);
    }
  }
  __syncthreads();
  const int r = t & (kToiLanes - 1);
  for (int k = t / kToiLanes; k < s_n; k += 256 / kToiLanes) {
    const int2 pr = s_body[k];
    unsigned long long key = kNoKey;
    float toi;
    if (pair_toi(b, c, pr.x, pr.y, -1.0f, -1.0f, dt0, target, on_penetration, r, &toi)) {
      if (!(toi > end_time)) key = toi_key(toi, s_pair[k]);
      else if (r == 0) atomicMin(&c.ctl[kCcdMinAfter], __float_as_uint(toi));  // toi > 0: the bits order as the values
    }
    if (r == 0) {
      c.key[s_first + uint32_t(k)] = key;
      if (key != kNoKey) c.ctl[kCcdAnyIn] = 1u;
    }
  }
}

// The CCD slots of every dynamic body (adjacency in slot order is not needed: the re-sweep's
// results go into the queue, whose order is by key), and the bodies that have any.
__global__ void __launch_bounds__(256) k_ccd_fill(int npairs, CcdBufs c) {
  const int slot = blockIdx.x * blockDim.x + threadIdx.x;
  if (slot >= npairs || slot >= int(c.ctl[kCcdSlots])) return;
  const int4 sb = c.slot_bodies[slot];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if ((h ? sb.w : sb.z) & kSlotStatic) continue;
    const int i = h ? sb.y : sb.x;
    const uint32_t k = atomicAdd(&c.fill[i], 1u);
    c.adj[c.off[i] + k] = slot;
    if (k == 0u) c.bodies[atomicAdd(&c.ctl[kCcdBodies], 1u)] = i;
  }
}

// ---- the impact queue ----
// Each CCD slot holds at most one key (its latest time of impact, kNoKey for none), so a re-sweep
// replaces it in place: no superseded entries to pop. The slots are cut into groups of 64 (more where
// that gives over kGroups) whose smallest keys live in LDS: the earliest of all is found by one wave among
// those, a key that falls is one LDS atomic, and only a group whose smallest key rose is
// searched again. Keys are unique (they hold the pair index): the order is total. It takes the place of an indexed 64-ary
// heap, whose updates one wave did one by one: see k_ccd_events.
constexpr int kGroups = kCcdGroups;

// Smallest value across the wave, in every lane: DPP steps within quads, half rows and rows, then
// row broadcasts; lane 63 ends with the minimum.
template <int Ctrl, int RowMask>
__device__ __forceinline__ uint32_t dpp_min_step(uint32_t v) {
  const uint32_t o = uint32_t(__builtin_amdgcn_update_dpp(int(v), int(v), Ctrl, RowMask, 0xf, false));
  return o < v ? o : v;
}
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
  v = dpp_min_step<0xb1, 0xf>(v);   // quad_perm [1,0,3,2]
  v = dpp_min_step<0x4e, 0xf>(v);   // quad_perm [2,3,0,1]
  v = dpp_min_step<0x141, 0xf>(v);  // row_half_mirror
  v = dpp_min_step<0x140, 0xf>(v);  // row_mirror
  v = dpp_min_step<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_min_step<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return uint32_t(__builtin_amdgcn_readlane(int(v), 63));
}

// The smallest of the wave's 64 keys (uniform): the time bits first, then the pair index among the
// lanes with that time.
__device__ __forceinline__ unsigned long long wave_min(unsigned long long k) {
  const uint32_t hi = uint32_t(k >> 32), lo = uint32_t(k & 0xffffffffull);
  const uint32_t mh = wave_min_u32(hi);
  const uint32_t ml = wave_min_u32(hi == mh ? lo : 0xffffffffu);
  return (static_cast<unsigned long long>(mh) << 32) | ml;
}

// The smallest key of slots [first, last) (uniform).
__device__ __forceinline__ unsigned long long range_min(const unsigned long long* key, int first, int last, int lane) {
  unsigned long long m = kNoKey;
  for (int k = first + lane; k < last; k += 64) m = key[k] < m ? key[k] : m;
  return wave_min(m);
}

// The times of impact that freezing a body at its earliest key would ask for, recorded per slot and side
// with that freeze time: a row of lanes per slot, a workgroup per body.
__global__ void __launch_bounds__(256) k_ccd_foresee(DevBodies b, CcdBufs c, float end_time, float target,
                                                     int on_penetration) {
  if (c.ctl[kCcdState] == kQueueDone || c.ctl[kCcdAnyIn] == 0u) return;
  const int t = threadIdx.x, lane = t & 63, r = t & (kToiLanes - 1);
  const int nb = int(c.ctl[kCcdBodies]);
  for (int at = blockIdx.x; at < nb; at += gridDim.x) {
    const int x = c.bodies[at];
    if (c.frozen[b.ccd_key[x]] >= 0.0f) continue;
    const int first = int(c.off[x]), n = int(c.deg[x]);
    unsigned long long m = kNoKey;
    for (int k = lane; k < n; k += 64) {
      const unsigned long long key = c.key[c.adj[first + k]];
      m = key < m ? key : m;
    }
    m = wave_min(m);
    if (m == kNoKey) continue;
    const float f = key_toi(m);
    for (int k = t / kToiLanes; k < n; k += 256 / kToiLanes) {
      const int slot = c.adj[first + k];
      const int4 sb = c.slot_bodies[slot];
      const int h = sb.x == x ? 0 : 1;
      const int other = h ? sb.z : sb.w;
      if ((other & kSlotStatic) || c.frozen[other] >= 0.0f || c.seen_at[2 * slot + h] == f) continue;
      float toi;
      const bool hit = pair_toi(b, c, sb.x, sb.y, h ? -1.0f : f, h ? f : -1.0f, end_time, target, on_penetration, r, &toi);
      if (r == 0) {
        c.seen_key[2 * slot + h] = hit ? toi_key(toi, c.slot_pair[slot]) : kNoKey;
        c.seen_at[2 * slot + h] = f;
      }
    }
  }
}

// Freeze times held in LDS for up to this many body keys (the rest of the 160 KB beside the groups).
constexpr int kFzCap = 27648;

// predict_next_impacts' event loop (mechanical_world.rs:453-557) in one workgroup, from where the last
// launch left it to the end of the window or the kEventMisses-th event with times not foreseen; with LdsFrozen
// the freeze times live in LDS meanwhile. What bounds it is the chain of events. With every re-sweep
// made in it, one query per lane, and a heap updated entry by entry, an event took 30-60 us (15-38 of re-sweep, the
// rest pops of keys that no longer counted and updates): 18.9 ms a step at 343 cuboids, 280 impacts and 9,000 pairs.
// Now some 25 events share a round of 30 us of k_ccd_foresee and 90 us here: 6.1 ms, with the substep.
template <bool LdsFrozen>
__global__ void __launch_bounds__(kEventBlock) k_ccd_events(DevBodies b, CcdBufs c, float end_time, float dt0,
                                                            float target, int on_penetration) {
  __shared__ unsigned long long s_min[kGroups];
  __shared__ float s_fz[LdsFrozen ? kFzCap : 1];
  __shared__ uint32_t s_bits[kGroups / 32];
  __shared__ uint16_t s_dirty[kGroups];
  __shared__ int s_go, s_i, s_j, s_fresh, s_nmiss, s_ndirty, s_nimp;
  float* const fz = LdsFrozen ? s_fz : c.frozen;
  constexpr int kKey = kSlotStatic - 1;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t state = c.ctl[kCcdState];
  if (state == kQueueDone) return;
  const int ns = int(c.ctl[kCcdSlots]);
  int sh = 6;
  while (((ns - 1) >> sh) >= kGroups) ++sh;
  const int ng = (ns + (1 << sh) - 1) >> sh;
  if (state == kQueueNew) {
    // min_overstep (mechanical_world.rs:412-451): the step's end lowered to the earliest impact
    // after the window, or the window's end when an impact lies within it
    const bool any = c.ctl[kCcdAnyIn] != 0u;
    float min_over = dt0;
    const float after = __uint_as_float(c.ctl[kCcdMinAfter]);
    if (after < min_over) min_over = after;
    if (any) min_over = end_time;
    int kind = PREDICT_IMPACTS;
    if (min_over == dt0 && !any) kind = PREDICT_NONE;
    else if (min_over > end_time) kind = PREDICT_AFTER_END;
    __syncthreads();
    if (t == 0) {
      c.ctl[kCcdKind] = uint32_t(kind);
      c.ctl[kCcdMinOver] = __float_as_uint(min_over);
      if (kind != PREDICT_IMPACTS) c.ctl[kCcdState] = kQueueDone;
    }
    if (kind != PREDICT_IMPACTS) return;
  }
  for (int g = wave; g < ng; g += kEventBlock / 64) {
    const unsigned long long m =
        state == kQueueNew ? range_min(c.key, g << sh, min((g + 1) << sh, ns), lane) : c.group[g];
    if (lane == 0) s_min[g] = m;
  }
  if (LdsFrozen)
    for (int k = t; k < b.n; k += kEventBlock) s_fz[k] = c.frozen[k];
  for (int k = t; k < kGroups / 32; k += kEventBlock) s_bits[k] = 0u;
  if (t == 0) {
    s_nimp = state == kQueueNew ? 0 : int(c.ctl[kCcdImpacts]);
    s_nmiss = s_ndirty = 0;
  }
  __syncthreads();
  // The slot's key, and its group's smallest: lowered at once, or noted to be searched again.
  auto set_key = [&](int slot, unsigned long long k) {
    const unsigned long long old = c.key[slot];
    if (k == old) return;
    c.key[slot] = k;
    const int g = slot >> sh;
    if (k < old) {
      atomicMin(&s_min[g], k);
    } else if (s_min[g] == old) {
      const uint32_t bit = 1u << (g & 31);
      if (!(atomicOr(&s_bits[g >> 5], bit) & bit)) s_dirty[atomicAdd(&s_ndirty, 1)] = uint16_t(g);
    }
  };
  int late = 0;  // events with times not foreseen
  for (;;) {
    // ---- wave 0 takes the earliest keys up to the next impact that freezes a body
    if (t < 64) {
      int nimp = s_nimp, go = 0;
      for (;;) {
        unsigned long long mine = kNoKey;
        int mg = 0;
        for (int g = lane; g < ng; g += 64) {
          const unsigned long long x = s_min[g];
          if (x < mine) {
            mine = x;
            mg = g;
          }
        }
        const unsigned long long ek = wave_min(mine);
        if (ek == kNoKey) break;
        if (nimp >= c.cap) {  // the impact list is full: reported as an overflow
          if (lane == 0) c.ctl[kCcdOverflow] = 1u;
          break;
        }
        const int g = __builtin_amdgcn_readlane(mg, __ffsll(static_cast<long long>(__ballot(mine == ek))) - 1);
        int es = 0;
        unsigned long long rest = kNoKey;
        for (int k = (g << sh) + lane; k - lane < min((g + 1) << sh, ns); k += 64) {
          const unsigned long long x = k < ns ? c.key[k] : kNoKey;
          const unsigned long long hit = __ballot(x == ek);
          if (hit) es = k - lane + __ffsll(static_cast<long long>(hit)) - 1;
          rest = (x != ek && x < rest) ? x : rest;
        }
        const int4 sb = c.slot_bodies[es];
        rest = wave_min(rest);
        if (lane == 0) {
          s_min[g] = rest;
          c.key[es] = kNoKey;
        }
        const float toi = key_toi(ek);
        const int ki = sb.z & kKey, kj = sb.w & kKey;
        const float t1 = fz[ki], t2 = fz[kj];
        if (t1 >= 0.0f && t2 >= 0.0f) {
          if (toi == (t1 > t2 ? t1 : t2)) {
            if (lane == 0) c.impacts[nimp] = ek;
            ++nimp;
          }
          continue;
        }
        if (lane == 0) {
          if (t1 < 0.0f) fz[ki] = toi;
          if (t2 < 0.0f) fz[kj] = toi;
          c.impacts[nimp] = ek;
          s_i = sb.x;
          s_j = sb.y;
          s_fresh = (t1 < 0.0f ? 1 : 0) | (t2 < 0.0f ? 2 : 0);
        }
        ++nimp;
        go = 1;
        break;
      }
      if (lane == 0) {
        s_nimp = nimp;
        s_go = go;
      }
    }
    __syncthreads();
    if (!s_go) break;
    // ---- re-sweep the CCD slots of the bodies' dynamic colliders (mechanical_world.rs:503-551); a body
    // frozen before has its slots' times already. A slot whose key no longer counts, its two bodies
    // being frozen at other times, is emptied; the event's own is empty.
    const int si = s_i, sj = s_j, fresh = s_fresh;
    const int ni = (fresh & 1) ? int(c.deg[si]) : 0;  // deg: 0 for a body that is not dynamic
    const int nj = (fresh & 2) ? int(c.deg[sj]) : 0;
    for (int k = t; k < ni + nj; k += kEventBlock) {
      const int slot = k < ni ? c.adj[c.off[si] + k] : c.adj[c.off[sj] + (k - ni)];
      const int4 sb = c.slot_bodies[slot];
      const float fa = fz[sb.z & kKey], fb = fz[sb.w & kKey];
      if (fa >= 0.0f && fb >= 0.0f) {
        const unsigned long long old = c.key[slot];
        if (old != kNoKey && key_toi(old) != (fa > fb ? fa : fb)) set_key(slot, kNoKey);
        continue;
      }
      if ((sb.z | sb.w) & kSlotStatic) continue;  // as it was: the static side moves no more than before
      const int h = fa >= 0.0f ? 0 : 1;
      if (c.seen_at[2 * slot + h] == (h ? fb : fa)) set_key(slot, c.seen_key[2 * slot + h]);
      else c.stage[atomicAdd(&s_nmiss, 1)] = slot;
    }
    __syncthreads();
    const int nmiss = s_nmiss;
    if (nmiss) {
      const int r = t & (kToiLanes - 1);
      for (int k = t / kToiLanes; k < nmiss; k += kEventBlock / kToiLanes) {
        const int slot = c.stage[k];
        const int4 sb = c.slot_bodies[slot];
        float toi;
        const bool hit = pair_toi(b, c, sb.x, sb.y, fz[sb.z & kKey], fz[sb.w & kKey], end_time, target, on_penetration,
                                  r, &toi);
        if (r == 0) set_key(slot, hit ? toi_key(toi, c.slot_pair[slot]) : kNoKey);
      }
      ++late;
      __syncthreads();
    }
    const int nd = s_ndirty;
    for (int k = wave; k < nd; k += kEventBlock / 64) {
      const int g = s_dirty[k];
      const unsigned long long m = range_min(c.key, g << sh, min((g + 1) << sh, ns), lane);
      if (lane == 0) {
        s_min[g] = m;
        s_bits[g >> 5] = 0u;
      }
    }
    __syncthreads();
    if (t == 0) s_nmiss = s_ndirty = 0;
    if (late >= kEventMisses) break;
  }
  __syncthreads();
  if (LdsFrozen)
    for (int k = t; k < b.n; k += kEventBlock) c.frozen[k] = s_fz[k];
  for (int g = t; g < ng; g += kEventBlock) c.group[g] = s_min[g];
  if (t == 0) {
    const int nimp = s_nimp;
    c.ctl[kCcdState] = s_go ? kQueueOpen : kQueueDone;
    c.ctl[kCcdImpacts] = uint32_t(nimp);
    c.ctl[kCcdLastToi] = nimp > 0 ? uint32_t(c.impacts[nimp - 1] >> 32) : 0u;
  }
}

__global__ void __launch_bounds__(256) k_ccd_island(int n, int P, CcdBufs c) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) c.in_t[i] = c.new_t[i] = c.prep[i] = c.prepared[i] = 0u;
  if (i < P) c.evaluated[i] = c.kept[i] = 0u;
}

__global__ void __launch_bounds__(256) k_ccd_seed(DevBodies b, const int2* __restrict__ pairs, CcdBufs c, int nimp) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nimp) return;
  const int2 pr = pairs[key_pair(c.impacts[k])];
  c.in_t[b.ccd_key[pr.x]] = 1u;
  c.in_t[b.ccd_key[pr.y]] = 1u;
}

__global__ void __launch_bounds__(256) k_ccd_touch(DevBodies b, const int2* __restrict__ pairs, int npairs,
                                                   CcdBufs c) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npairs) return;
  const int2 pr = pairs[p];
  const bool on = !c.evaluated[p] && (c.in_t[b.ccd_key[pr.x]] || c.in_t[b.ccd_key[pr.y]]);
  c.cand[p] = on ? 1u : 0u;
  if (!on) return;
  if (b.status[pr.x] == STATUS_DYNAMIC) c.prep[pr.x] = 1u;
  if (b.status[pr.y] == STATUS_DYNAMIC) c.prep[pr.y] = 1u;
}

// prepare_body (mechanical_world.rs:653-681): forces cleared, the dynamics update of the substep
// (dt_sub, no gravity) at the current pose, then RigidBody::advance to the body's freeze time (or
// the last impact time) along its motion and clamp_advancement.
__global__ void __launch_bounds__(256) k_ccd_prepare(DevBodies b, CcdBufs c, float dt_sub, float last_toi) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= b.n || !c.prep[i] || c.prepared[i]) return;
  c.prepared[i] = 1u;
  if (b.f_lin) {
    b.f_lin[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    b.f_ang[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  body_prestep(b, i, toq(b.rot(i)), xyz(b.angvel[i]), false, false, f3{0.0f, 0.0f, 0.0f}, dt_sub, dt_sub,
               f3{0.0f, 0.0f, 0.0f});
  const float f = c.frozen[b.ccd_key[i]];
  const float target = f >= 0.0f ? f : last_toi;
  const CcdMotion m = part_motion(b, i, 0.0f);
  f3 tp;
  q4 q;
  m.at(target - c.body_time[i], tp, q);
  b.pos0[i] = f4(tp, 0.0f);
  b.rot0[i] = fromq(q);
  b.pos(i) = f4(tp, 0.0f);
  if (!(b.ccd[i] & 2)) b.rot(i) = fromq(q);
  c.body_time[i] = last_toi;
}

__global__ void __launch_bounds__(256) k_ccd_scatter(const int2* __restrict__ pairs, int npairs,
                                                     const uint32_t* __restrict__ flag, CcdBufs c) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npairs) return;
  const uint32_t at = c.cpos[p];
  if (p == npairs - 1) c.ctl[kCcdList] = at + flag[p];
  if (!flag[p]) return;
  c.list[at] = pairs[p];
  c.list_pair[at] = p;
}

__global__ void __launch_bounds__(256) k_ccd_grow(DevBodies b, CcdBufs c, int nlist, const uint32_t* __restrict__ count) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nlist) return;
  const int p = c.list_pair[k];
  c.evaluated[p] = 1u;
  if (count[k] == 0u) return;
  c.kept[p] = 1u;
  const int2 pr = c.list[k];
  if (b.status[pr.x] == STATUS_DYNAMIC && !c.in_t[b.ccd_key[pr.x]]) c.new_t[b.ccd_key[pr.x]] = 1u;
  if (b.status[pr.y] == STATUS_DYNAMIC && !c.in_t[b.ccd_key[pr.y]]) c.new_t[b.ccd_key[pr.y]] = 1u;
}

__global__ void __launch_bounds__(256) k_ccd_merge(int n, CcdBufs c) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !c.new_t[i]) return;
  c.in_t[i] = 1u;
  c.new_t[i] = 0u;
}

__global__ void __launch_bounds__(256) k_ccd_validate(DevBodies b, const int2* __restrict__ pairs, CcdBufs c, int nimp) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nimp) return;
  const int2 pr = pairs[key_pair(c.impacts[k])];
  if (b.status[pr.x] == STATUS_DYNAMIC) {
    b.pos0[pr.x] = b.pos(pr.x);
    b.rot0[pr.x] = b.rot(pr.x);
  }
  if (b.status[pr.y] == STATUS_DYNAMIC) {
    b.pos0[pr.y] = b.pos(pr.y);
    b.rot0[pr.y] = b.rot(pr.y);
  }
}

// The bodies still frozen when the CCD ends go back to their safe position; their last dynamics
// update (after the substep) used the rotation they have now, kept for the next one.
__global__ void __launch_bounds__(256) k_ccd_clamp(DevBodies b, CcdBufs c) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= b.n || b.status[i] != STATUS_DYNAMIC || !(c.frozen[b.ccd_key[i]] >= 0.0f)) return;
  b.ccd_rot[i] = b.rot(i);
  b.w_dyn[i].w = 2.0f;
  b.pos(i) = b.pos0[i];
  if (!(b.ccd[i] & 2)) b.rot(i) = b.rot0[i];
}

int blocks_of(int n, int bs) { return (n + bs - 1) / bs; }

}  // namespace

void launch_ccd_first(const DevBodies& b, const int2* pairs, int npairs, CcdBufs& c, float end_time, float dt0,
                      float target, int on_penetration, hipStream_t s) {
  hipLaunchKernelGGL(k_ccd_begin, dim3(blocks_of(std::max(b.n, int(kCcdWords)), 256)), dim3(256), 0, s, b.n, c);
  if (npairs <= 0) return;
  hipLaunchKernelGGL(k_ccd_first_pass, dim3(blocks_of(npairs, kFirstPairs)), dim3(256), 0, s, b, pairs, npairs, c,
                     end_time, dt0, target, on_penetration);
  scan_exclusive_u32(c.deg, c.off, b.n, *c.scan, s);
  hipLaunchKernelGGL(k_ccd_fill, dim3(blocks_of(npairs, 256)), dim3(256), 0, s, npairs, c);
}

void launch_ccd_events(const DevBodies& b, CcdBufs& c, float end_time, float dt0, float target, int on_penetration,
                       hipStream_t s) {
  hipLaunchKernelGGL(k_ccd_foresee, dim3(std::min(std::max(b.n, 1), 4096)), dim3(256), 0, s, b, c, end_time, target,
                     on_penetration);
  if (b.n <= kFzCap)
    hipLaunchKernelGGL(k_ccd_events<true>, dim3(1), dim3(kEventBlock), 0, s, b, c, end_time, dt0, target,
                       on_penetration);
  else
    hipLaunchKernelGGL(k_ccd_events<false>, dim3(1), dim3(kEventBlock), 0, s, b, c, end_time, dt0, target,
                       on_penetration);
}

void launch_ccd_island(int n, int P, CcdBufs& c, hipStream_t s) {
  hipLaunchKernelGGL(k_ccd_island, dim3(blocks_of(std::max(n, P), 256)), dim3(256), 0, s, n, P, c);
}

void launch_ccd_seed(const DevBodies& b, const int2* pairs, CcdBufs& c, int nimp, hipStream_t s) {
  if (nimp <= 0) return;
  hipLaunchKernelGGL(k_ccd_seed, dim3(blocks_of(nimp, 256)), dim3(256), 0, s, b, pairs, c, nimp);
}

void launch_ccd_touch(const DevBodies& b, const int2* pairs, int npairs, CcdBufs& c, hipStream_t s) {
  if (npairs <= 0) return;
  hipLaunchKernelGGL(k_ccd_touch, dim3(blocks_of(npairs, 256)), dim3(256), 0, s, b, pairs, npairs, c);
}

void launch_ccd_prepare(const DevBodies& b, CcdBufs& c, float dt_sub, float last_toi, hipStream_t s) {
  if (b.n <= 0) return;
  hipLaunchKernelGGL(k_ccd_prepare, dim3(blocks_of(b.n, 256)), dim3(256), 0, s, b, c, dt_sub, last_toi);
}

void launch_ccd_compact(const int2* pairs, int npairs, const uint32_t* flag, CcdBufs& c, hipStream_t s) {
  if (npairs <= 0) {
    fill_u32(c.ctl + kCcdList, 0u, 1, s);
    return;
  }
  scan_exclusive_u32(flag, c.cpos, npairs, *c.scan, s);
  hipLaunchKernelGGL(k_ccd_scatter, dim3(blocks_of(npairs, 256)), dim3(256), 0, s, pairs, npairs, flag, c);
}

void launch_ccd_grow(const DevBodies& b, CcdBufs& c, int nlist, const uint32_t* count, hipStream_t s) {
  if (nlist <= 0) return;
  hipLaunchKernelGGL(k_ccd_grow, dim3(blocks_of(nlist, 256)), dim3(256), 0, s, b, c, nlist, count);
}

void launch_ccd_merge(int n, CcdBufs& c, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_ccd_merge, dim3(blocks_of(n, 256)), dim3(256), 0, s, n, c);
}

void launch_ccd_validate(const DevBodies& b, const int2* pairs, CcdBufs& c, int nimp, hipStream_t s) {
  if (nimp <= 0) return;
  hipLaunchKernelGGL(k_ccd_validate, dim3(blocks_of(nimp, 256)), dim3(256), 0, s, b, pairs, c, nimp);
}

void launch_ccd_clamp(const DevBodies& b, CcdBufs& c, hipStream_t s) {
  if (b.n <= 0) return;
  hipLaunchKernelGGL(k_ccd_clamp, dim3(blocks_of(b.n, 256)), dim3(256), 0, s, b, c);
}

}  // namespace nph
