// nphysics_amd/csrc/k_solver.hip -- contact assembly and the graph-coloured SOR-Prox solve.
//
// Colouring. Manifolds conflict when they share a dynamic body. A deterministic Jones-Plassmann
// greedy colouring runs one kernel per round: every uncoloured manifold whose priority
// (hash(m), m) beats all neighbours that are uncoloured or were coloured in this same round takes
// the smallest colour unused by neighbours coloured in earlier rounds. The state word packs
// (round << 16 | colour), so a neighbour coloured concurrently in the current round is always
// seen as "this round" whichever value the load returns; the result is independent of timing.
// Colours persist across steps: manifolds whose body pair was solved in the previous step keep
// their colour and only new manifolds run the rounds, so at rest colouring costs one pass.
// Manifolds are then put in colour order by a stable counting sort and row records laid out in that order.
//
// Assembly (k_assemble, one lane per manifold) restates SignoriniCoulombPyramidModel::constraints
// (src/solver/signorini_coulomb_pyramid_model.rs:56-224), SignoriniModel::build_velocity_constraint
// (src/solver/signorini_model.rs:37-138), helper::constraint_pair_geometry
// (src/solver/helper.rs:53-135) and RigidBody::fill_constraint_geometry
// (src/object/rigid_body.rs:672-722): per contact one normal row along -n at
// world1 + n margin1 / world2 - n margin2 and two friction rows along the tangents; material
// Average combine (src/material/material.rs:72-86); warm start from the previous step's impulse
// of the contact with the same (body1, body2, feature) key (the ImpulseCache lookup at
// signorini_coulomb_pyramid_model.rs:104-108).
//
// Solve (k_pgs) restates SORProx (src/solver/sor_prox.rs:19-436): warm start dv += l W J,
// then per sweep and contact the normal row (projected on l >= 0) and the two friction rows (bounded by
// mu times the normal impulse just computed, zeroed when it is zero). Manifolds of one colour share no
// dynamic body, so one launch per colour performs exactly the sequential Gauss-Seidel updates of
// the colour order. A contact has two adjacent lanes, one per body (ContactLane): a lane loads its body's
// inverse inertia and the contact, forms its body's half of the three rows at once, and then the
// manifold's contacts take their turns, the velocity increments handed from one pair of lanes to the
// next and the halves of J dv exchanged within the pair, both by register permutations. A class lists the manifolds with
// several contacts first: those have four pairs of lanes each, the others one.
//
// Row record (4 contiguous float4 per contact, colour order): 0 n|length of the tangents' seed, 1 lever arm
// p1 of body 1 (contact point minus centre of mass, zero for a static body)|r_n, 2 p2|r_t1,
// 3 rhs (n, t1, t2)|r_t2. The impulses live in their own array, one float4 per record (n, t1, t2
// | mu), so a sweep's impulse writes are contiguous 16-byte runs rather than one dirty line per
// contact. What the sweeps spend their time on is instructions, one wave per SIMD or two: the seed's
// length saves them a square root and (a quotient per lane) two of three divisions per contact.
// Linear jacobians are the row direction d (body 1) and -d (body 2) weighted by the inverse
// mass; the tangents, the angular jacobians p1 x d and p2 x (-d) and I^-1 J_ang are recomputed
// in the sweep kernels with the assembly's own expressions, so they carry the same FP32 values.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include "kernels.hpp"
#include "stages.hpp"

namespace nph {

namespace {

constexpr uint32_t kUncoloured = 0xffffffffu;

__device__ __forceinline__ uint32_t colour_hash(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352dU;
  x ^= x >> 15;
  x *= 0x846ca68bU;
  x ^= x >> 16;
  return x;
}

// Colours persist across steps: a manifold whose body pair was a manifold of the previous solve
// keeps that colour (marked as coloured in round 0); the others start uncoloured. Also counts the
// manifolds of every dynamic body; the count met is the manifold's place in that body's list.
constexpr uint32_t kNoPlace = 0xffffffffu;  // the static side of a manifold

__global__ void __launch_bounds__(256) k_colour_begin(DevBodies b, DevContacts c, int M, DevContacts prev, int prevM,
                                                     const uint32_t* __restrict__ prev_state, SolverBufs sb) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  const int2 bb = c.mbody[m];
  uint2 at = make_uint2(kNoPlace, kNoPlace);
  if (b.status[bb.x] == STATUS_DYNAMIC) at.x = atomicAdd(&sb.deg[bb.x], 1u);
  if (b.status[bb.y] == STATUS_DYNAMIC) at.y = atomicAdd(&sb.deg[bb.y], 1u);
  sb.place[m] = at;
  const int j = find_manifold(prev, prevM, bb.x, bb.y);
  sb.state[m] = j >= 0 ? (prev_state[j] & 0xffffu) : kUncoloured;
}

__global__ void __launch_bounds__(256) k_adjacency(DevContacts c, int M, SolverBufs sb) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  const int2 bb = c.mbody[m];
  const uint2 at = sb.place[m];
  if (at.x != kNoPlace) sb.adj[sb.adj_off[bb.x] + at.x] = m;
  if (at.y != kNoPlace) sb.adj[sb.adj_off[bb.y] + at.y] = m;
}

// kLanes 1: a lane per manifold; kLanes 16: a row of lanes per manifold, over its neighbours. What bounds a
// round is the chain of loads (neighbour, then its state) of the longest lists: see launch_colour_round.
template <int kLanes>
__device__ __forceinline__ bool row_any(bool x) {
  if (kLanes == 1) return x;
  return ((__ballot(x) >> (threadIdx.x & 48)) & 0xffffull) != 0ull;
}

template <int kLanes>
__global__ void __launch_bounds__(256) k_colour_round(DevContacts c, int M, uint32_t round,
                                                     const uint32_t* __restrict__ off,
                                                     const uint32_t* __restrict__ deg,
                                                     const int* __restrict__ adj, const uint2* __restrict__ place,
                                                     uint32_t* state, uint32_t* remaining, uint32_t* last_round) {
  const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
  const long mm = t / kLanes;
  const uint32_t r = uint32_t(t % kLanes);
  if (mm >= M) return;
  const int m = int(mm);
  if (state[m] != kUncoloured) return;
  const uint32_t pm = colour_hash(uint32_t(m));
  const int2 bb = c.mbody[m];
  const uint2 at = place[m];
  const uint32_t n1 = at.x != kNoPlace ? deg[bb.x] : 0u, n2 = at.y != kNoPlace ? deg[bb.y] : 0u;
  const uint32_t o1 = off[bb.x], o2 = off[bb.y];
  const uint32_t n = n1 + n2, up = (n + kLanes - 1) / kLanes * kLanes;  // the lanes of a row go on together
  auto neighbour = [&](uint32_t k) { return adj[k < n1 ? o1 + k : o2 + (k - n1)]; };
  for (uint32_t k = r; k < up; k += kLanes) {
    bool before = false;  // a neighbour not coloured before this round whose turn comes first
    if (k < n) {
      const int o = neighbour(k);
      if (o != m) {
        const uint32_t so = state[o];
        if (so == kUncoloured || (so >> 16) == round) {
          const uint32_t po = colour_hash(uint32_t(o));
          before = po > pm || (po == pm && o > m);
        }
      }
    }
    if (row_any<kLanes>(before)) {
      *remaining = 1u;  // any uncoloured manifold left; a plain store, every writer stores 1
      return;
    }
  }
  uint32_t colour = 0;
  for (uint32_t base = 0;; base += 64) {
    uint64_t mask = 0;
    for (uint32_t k = r; k < n; k += kLanes) {
      const int o = neighbour(k);
      if (o == m) continue;
      const uint32_t so = state[o];
      if (so == kUncoloured || (so >> 16) == round) continue;
      const uint32_t cc = so & 0xffffu;
      if (cc >= base && cc < base + 64) mask |= 1ull << (cc - base);
    }
    if (kLanes > 1) {
#pragma unroll
      for (int x = 1; x < 16; x <<= 1) mask |= __shfl_xor(static_cast<unsigned long long>(mask), x, 16);
    }
    if (mask != ~0ull) {
      colour = base + uint32_t(__ffsll((long long)(~mask))) - 1u;
      break;
    }
  }
  if (r != 0u) return;
  state[m] = (round << 16) | colour;
  atomicMax(last_round, round);
}

// Colour order: a stable counting sort of the manifolds by colour that also adds up their contacts,
// so that a manifold's slot, its first row record and the classes' bounds come out of one prefix sum over
// (manifolds per colour and tile, then contacts per colour and tile). k_colour_hist counts per tile of
// kColourTile manifolds, k_colour_scatter ranks within its tile: lanes of equal colour find each other by
// ballots, and three ballots more give the contacts of those before. kDigits at most (512, or
// kMaxColours where a readback finds more colours); a colour beyond, or none yet, counts as the last, and the
// caller runs it again. The sort by a radix pass (histogram, scan, scatter, two copies back), the class starts, the
// gather and scan of the counts, the slot records and the fix of empty classes were 14 launches and
// one readback more: 30 us of a step at 1,233 manifolds, now 13 us.
//
// With kSplit a class lists its manifolds with several contacts before those with one, so that the
// sweeps can give them different numbers of lanes: a digit is then 2 colour + (one contact).
constexpr int kColourTile = 2048;

template <int kDigits, bool kSplit>
__device__ __forceinline__ uint32_t colour_digit(uint32_t state, uint32_t contacts) {
  const uint32_t c = state & 0xffffu, d = kSplit ? 2u * c + (contacts == 1u ? 1u : 0u) : c;
  return d < uint32_t(kDigits) ? d : uint32_t(kDigits) - 1u;
}

template <int kDigits, int kThreads, bool kSplit>
__global__ void __launch_bounds__(kThreads) k_colour_hist(DevContacts c, int M, int ntiles, SolverBufs sb,
                                                         uint32_t* ncol) {
  __shared__ uint32_t s_m[kDigits], s_c[kDigits];
  __shared__ uint32_t s_most;
  for (int d = threadIdx.x; d < kDigits; d += kThreads) s_m[d] = s_c[d] = 0u;
  if (threadIdx.x == 0) s_most = 0u;
  __syncthreads();
  uint32_t most = 0;
  for (int k = threadIdx.x; k < kColourTile; k += kThreads) {
    const int m = int(blockIdx.x) * kColourTile + k;
    if (m >= M) break;
    const uint32_t st = sb.state[m];
    const uint32_t cnt = uint32_t(c.mcount[m]);
    const uint32_t d = colour_digit<kDigits, kSplit>(st, cnt);
    const uint32_t c1 = (st & 0xffffu) + 1u;
    most = c1 > most ? c1 : most;
    atomicAdd(&s_m[d], 1u);
    atomicAdd(&s_c[d], cnt);
  }
  atomicMax(&s_most, most);
  __syncthreads();
  for (int d = threadIdx.x; d < kDigits; d += kThreads) {
    sb.hist[long(d) * ntiles + blockIdx.x] = s_m[d];
    sb.hist[long(kDigits + d) * ntiles + blockIdx.x] = s_c[d];
  }
  if (threadIdx.x == 0) atomicMax(ncol, s_most);
}

// The manifolds of the tile at `base` into their slots; s_m, s_c: the digits' first slots and records in this tile.
template <int kDigits, int kThreads, bool kSplit>
__device__ void scatter_tile(const DevContacts& c, int M, int base, const SolverBufs& sb, uint32_t* s_m, uint32_t* s_c,
                             uint32_t (*s_wave)[kDigits]) {
  constexpr int kWaves = kThreads / 64;
  constexpr int kBits = kDigits == 512 ? 9 : 12;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const uint64_t below = (1ull << lane) - 1ull;
  for (int k = 0; k < kColourTile; k += kThreads) {
    const int m = base + k + tid;
    if (base + k >= M) break;
    const bool valid = m < M;
    const uint32_t cnt = valid ? uint32_t(c.mcount[m]) : 0u;
    const uint32_t d = valid ? colour_digit<kDigits, kSplit>(sb.state[m], cnt) : 0u;
    uint64_t same = __ballot(valid);
#pragma unroll
    for (int i = 0; i < kBits; ++i) {
      const bool bit = (d >> i) & 1u;
      const uint64_t bb = __ballot(bit);
      same &= bit ? bb : ~bb;
    }
    const uint64_t c0 = __ballot(cnt & 1u), c1 = __ballot(cnt & 2u), c2 = __ballot(cnt & 4u);
    auto contacts = [&](uint64_t of) {
      return uint32_t(__popcll(of & c0) + 2 * __popcll(of & c1) + 4 * __popcll(of & c2));
    };
    if (valid && (same & below) == 0ull) s_wave[wave][d] = uint32_t(__popcll(same)) | (contacts(same) << 16);
    __syncthreads();
    if (valid) {
      uint32_t before = 0;
      for (int w = 0; w < wave; ++w) before += s_wave[w][d];
      const uint32_t slot = s_m[d] + (before & 0xffffu) + uint32_t(__popcll(same & below));
      const uint32_t r0 = s_c[d] + (before >> 16) + contacts(same & below);
      const int2 bb = c.mbody[m];
      const uint2 at = sb.place[m];
      sb.sinfo[slot] = make_int4(bb.x | (at.x != kNoPlace ? 1 << 30 : 0), bb.y | (at.y != kNoPlace ? 1 << 30 : 0),
                                 int(r0), int(cnt) | (c.mfirst[m] << 3));
      sb.ckeys[slot] = d;
      sb.slot_of[m] = make_uint2(slot, r0);
    }
    __syncthreads();
    for (int i = tid; i < kDigits; i += kThreads) {
      uint32_t all = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        all += s_wave[w][i];
        s_wave[w][i] = 0u;
      }
      s_m[i] += all & 0xffffu;
      s_c[i] += all >> 16;
    }
    __syncthreads();
  }
}

// Per slot (colour order): bodies with their dynamic flag in bit 30, first row record, contact
// count and first contact index, packed into one int4; per manifold its slot and first row record; per
// class its first slot and first row record (col_start, class_rec; one more entry ends the last).
template <int kDigits, int kThreads, bool kSplit>
__global__ void __launch_bounds__(kThreads) k_colour_scatter(DevContacts c, int M, int C, int ntiles, SolverBufs sb) {
  constexpr int kWaves = kThreads / 64;
  __shared__ uint32_t s_m[kDigits], s_c[kDigits];
  __shared__ uint32_t s_wave[kWaves][kDigits];  // per wave: manifolds, and their contacts from bit 16 up
  const int tid = threadIdx.x;
  for (int d = tid; d < kDigits; d += kThreads) {
    s_m[d] = sb.offs[long(d) * ntiles + blockIdx.x];
    s_c[d] = sb.offs[long(kDigits + d) * ntiles + blockIdx.x] - uint32_t(M);
    if (blockIdx.x == 0) {
      sb.col_start[d] = s_m[d];
      sb.class_rec[d] = s_c[d];
    }
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s_wave[w][d] = 0u;
  }
  if (blockIdx.x == 0 && tid == 0) {
    sb.col_start[kDigits] = uint32_t(M);
    sb.class_rec[kDigits] = uint32_t(C);
  }
  __syncthreads();
  scatter_tile<kDigits, kThreads, kSplit>(c, M, int(blockIdx.x) * kColourTile, sb, s_m, s_c, s_wave);
}

// ---- colouring and colour order of a small world in one workgroup ----
// Degrees, adjacency, rounds and order with the graph in LDS: the same states, colours and slots as the
// kernels above give, whose thirteen dependent launches of 2 to 8 us each a world of this size spends its time on:
// assembly stage 64 -> 45 us at 1,233 manifolds, 59 -> 39 at 320. Its one lane per manifold reads its
// neighbours one after another, so with a body of more than kSmallDegree manifolds it leaves the rounds to
// k_colour_round: in a cloud where all bodies touch, every round of some 60 to 200 waits for the longest list (24
// bodies: 689 us here, 731 there; 45: 3,096 and 1,726).
constexpr int kSmallThreads = 1024;
constexpr uint32_t kSmallDegree = 24;

// Exclusive sum over the workgroup's threads (uses s_tot, and ends on a barrier).
__device__ __forceinline__ uint32_t block_exclusive(uint32_t v, uint32_t* s_tot) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  if (lane == 63) s_tot[wave] = x;
  __syncthreads();
  uint32_t before = 0;
  for (int w = 0; w < wave; ++w) before += s_tot[w];
  __syncthreads();
  return before + x - v;
}

template <bool kSplit>
__global__ void __launch_bounds__(kSmallThreads) k_colour_small(DevBodies b, DevContacts c, int M, int C, DevContacts prev,
                                                              int prevM, const uint32_t* __restrict__ prev_state,
                                                              SolverBufs sb, uint32_t* words) {
  constexpr int kEach = kSmallManifolds / kSmallThreads;
  constexpr int kBodies = kSmallColourBodies / kSmallThreads;
  __shared__ uint32_t s_state[kSmallManifolds];
  __shared__ uint32_t s_deg[kSmallColourBodies], s_off[kSmallColourBodies];
  __shared__ uint16_t s_adj[2 * kSmallManifolds];
  __shared__ uint32_t s_m[kColourDigits], s_c[kColourDigits];
  __shared__ uint32_t s_wave[kSmallThreads / 64][kColourDigits];
  __shared__ uint32_t s_tot[kSmallThreads / 64];
  __shared__ uint32_t s_left[2], s_last, s_most, s_crowd;
  const int tid = threadIdx.x;
  for (int i = tid; i < kSmallColourBodies; i += kSmallThreads) s_deg[i] = 0u;
  if (tid == 0) s_left[0] = s_left[1] = s_last = s_most = s_crowd = 0u;
  __syncthreads();
  int2 bb[kEach];
  uint2 at[kEach];
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    const int m = tid + kSmallThreads * e;
    bb[e] = make_int2(0, 0);
    at[e] = make_uint2(kNoPlace, kNoPlace);
    if (m >= M) continue;
    bb[e] = c.mbody[m];
    if (b.status[bb[e].x] == STATUS_DYNAMIC) at[e].x = atomicAdd(&s_deg[bb[e].x], 1u);
    if (b.status[bb[e].y] == STATUS_DYNAMIC) at[e].y = atomicAdd(&s_deg[bb[e].y], 1u);
    sb.place[m] = at[e];
    const int j = find_manifold(prev, prevM, bb[e].x, bb[e].y);
    s_state[m] = j >= 0 ? (prev_state[j] & 0xffffu) : kUncoloured;
  }
  __syncthreads();
  {
    uint32_t sum = 0, most = 0;
    for (int i = 0; i < kBodies; ++i) {
      const uint32_t d = s_deg[tid * kBodies + i];
      sum += d;
      most = d > most ? d : most;
    }
    if (most > kSmallDegree) s_crowd = 1u;
    uint32_t off = block_exclusive(sum, s_tot);
    for (int i = 0; i < kBodies; ++i) {
      s_off[tid * kBodies + i] = off;
      off += s_deg[tid * kBodies + i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    const int m = tid + kSmallThreads * e;
    if (at[e].x != kNoPlace) s_adj[s_off[bb[e].x] + at[e].x] = uint16_t(m);
    if (at[e].y != kNoPlace) s_adj[s_off[bb[e].y] + at[e].y] = uint16_t(m);
  }
  __syncthreads();
  const bool crowd = s_crowd != 0u;
  if (crowd) {  // the graph for k_colour_round
    for (int i = tid; i < b.n; i += kSmallThreads) {
      sb.deg[i] = s_deg[i];
      sb.adj_off[i] = s_off[i];
    }
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const int m = tid + kSmallThreads * e;
      if (at[e].x != kNoPlace) sb.adj[s_off[bb[e].x] + at[e].x] = m;
      if (at[e].y != kNoPlace) sb.adj[s_off[bb[e].y] + at[e].y] = m;
    }
  }
  // the rounds of k_colour_round; the first manifold in priority is coloured in each, so M rounds end it
  for (uint32_t round = 1; !crowd && round <= uint32_t(M); ++round) {
    uint32_t* left = &s_left[round & 1u];
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const int m = tid + kSmallThreads * e;
      if (m >= M || s_state[m] != kUncoloured) continue;
      const uint32_t pm = colour_hash(uint32_t(m));
      const uint32_t n1 = at[e].x != kNoPlace ? s_deg[bb[e].x] : 0u, n2 = at[e].y != kNoPlace ? s_deg[bb[e].y] : 0u;
      const uint32_t o1 = s_off[bb[e].x], o2 = s_off[bb[e].y];
      const uint32_t n = n1 + n2;
      bool wait = false;
      uint64_t mask = 0;  // colours 0-63 of the neighbours coloured before this round
      for (uint32_t k = 0; k < n && !wait; ++k) {
        const int o = int(s_adj[k < n1 ? o1 + k : o2 + (k - n1)]);
        if (o == m) continue;
        const uint32_t so = s_state[o];
        if (so == kUncoloured || (so >> 16) == round) {
          const uint32_t po = colour_hash(uint32_t(o));
          wait = po > pm || (po == pm && o > m);
        } else {
          const uint32_t cc = so & 0xffffu;
          if (cc < 64u) mask |= 1ull << cc;
        }
      }
      if (wait) {
        *left = 1u;
        continue;
      }
      uint32_t colour = 0;
      for (uint32_t base = 0;; base += 64) {
        if (base > 0u) {
          mask = 0;
          for (uint32_t k = 0; k < n; ++k) {
            const int o = int(s_adj[k < n1 ? o1 + k : o2 + (k - n1)]);
            if (o == m) continue;
            const uint32_t so = s_state[o];
            if (so == kUncoloured || (so >> 16) == round) continue;
            const uint32_t cc = so & 0xffffu;
            if (cc >= base && cc < base + 64) mask |= 1ull << (cc - base);
          }
        }
        if (mask != ~0ull) {
          colour = base + uint32_t(__ffsll((long long)(~mask))) - 1u;
          break;
        }
      }
      s_state[m] = (round << 16) | colour;
      s_last = round;  // every writer of a round stores the same
    }
    __syncthreads();
    const bool more = *left != 0u;
    if (tid == 0) s_left[(round & 1u) ^ 1u] = 0u;
    __syncthreads();
    if (!more) break;
  }
  // the order
  for (int d = tid; d < kColourDigits; d += kSmallThreads) {
    s_m[d] = s_c[d] = 0u;
    for (int w = 0; w < kSmallThreads / 64; ++w) s_wave[w][d] = 0u;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    const int m = tid + kSmallThreads * e;
    if (m >= M) continue;
    const uint32_t st = s_state[m], cnt = uint32_t(c.mcount[m]);
    sb.state[m] = st;
    const uint32_t d = colour_digit<kColourDigits, kSplit>(st, cnt);
    atomicAdd(&s_m[d], 1u);
    atomicAdd(&s_c[d], cnt);
    atomicMax(&s_most, (st & 0xffffu) + 1u);
  }
  __syncthreads();
  const uint32_t vm = tid < kColourDigits ? s_m[tid] : 0u, vc = tid < kColourDigits ? s_c[tid] : 0u;
  const uint32_t em = block_exclusive(vm, s_tot), ec = block_exclusive(vc, s_tot);
  if (tid < kColourDigits) {
    s_m[tid] = em;
    s_c[tid] = ec;
    sb.col_start[tid] = em;
    sb.class_rec[tid] = ec;
  }
  if (tid == 0) {
    sb.col_start[kColourDigits] = uint32_t(M);
    sb.class_rec[kColourDigits] = uint32_t(C);
    words[0] = 0u;
    words[1] = crowd ? 1u : 0u;
    words[2] = s_most;
    words[3] = s_last;
  }
  __syncthreads();  // also sb.state and sb.place, which the tiles read again
  for (int base = 0; base < M; base += kColourTile)
    scatter_tile<kColourDigits, kSmallThreads, kSplit>(c, M, base, sb, s_m, s_c, s_wave);
}

// One fill_constraint_geometry call: body-side jacobian (dir, p x dir), weighted angular part,
// inv_r and rhs accumulation with J.v then J.ext.
struct BodyView {
  f3 com, v, w, el, ea;
  f3 ml, ma;  // jacobian mask
  m33 inv;
  float im;
};

// The jacobian [dir; p x dir] is masked; the velocity term uses the unmasked force, so kinematic
// dofs stay controllable at the velocity level, and the external term the masked one
// (rigid_body.rs:685-718).
__device__ __forceinline__ void fill_geom(const BodyView& bv, f3 point, f3 dir, f3& ang, f3& wang,
                                          float& inv_r, float& rhs) {
  const f3 p = sub(point, bv.com);
  const f3 ang_u = cross(p, dir);
  const f3 lin = cmul(dir, bv.ml);
  ang = cmul(ang_u, bv.ma);
  wang = mulv(bv.inv, ang);
  inv_r = inv_r + (bv.im + dot(ang, wang));
  const float F[6] = {dir.x, dir.y, dir.z, ang_u.x, ang_u.y, ang_u.z};
  const float J[6] = {lin.x, lin.y, lin.z, ang.x, ang.y, ang.z};
  const float V[6] = {bv.v.x, bv.v.y, bv.v.z, bv.w.x, bv.w.y, bv.w.z};
  const float E[6] = {bv.el.x, bv.el.y, bv.el.z, bv.ea.x, bv.ea.y, bv.ea.z};
  float s = 0.0f;
#pragma unroll
  for (int k = 0; k < 6; ++k) s = s + F[k] * V[k];
  rhs = rhs + s;
  float e = 0.0f;
#pragma unroll
  for (int k = 0; k < 6; ++k) e = e + J[k] * E[k];
  rhs = rhs + e;
}

__device__ __forceinline__ BodyView load_body(const DevBodies& b, int i) {
  BodyView v;
  v.com = xyz(b.pos(i));
  v.v = xyz(b.linvel[i]);
  v.w = xyz(b.angvel[i]);
  v.el = xyz(b.ext_lin[i]);
  v.ea = xyz(b.ext_ang[i]);
  v.inv = load_inv(b, i, v.im);
  b.mask(i, v.ml, v.ma);
  return v;
}

// The tangents' seed: a vector orthogonal to n with one zero component, of length l.
__device__ __forceinline__ f3 tangent_seed(f3 n) {
  return fabsf(n.x) > fabsf(n.y) ? f3{n.z, 0.0f, -n.x} : f3{0.0f, -n.z, n.y};
}

__device__ __forceinline__ void tangents(f3 n, float l, f3& t1, f3& t2) {
  f3 a = tangent_seed(n);
  a = f3{a.x / l, a.y / l, a.z / l};
  t1 = cross(a, n);
  t2 = a;
}

// Material::combine (material.rs:134-178): the table's coefficient when both materials have an
// id and the table holds the pair, else MaterialCombineMode::combine of the two.
__device__ __forceinline__ void material_coefficients(const DevBodies& b, const MatTable& mt, int b1, int b2,
                                                      float& mu, float& e) {
  const int f1 = b.flags ? b.flags[b1] : 0, f2 = b.flags ? b.flags[b2] : 0;
  mu = combine_coeff(b.friction[b1], fric_mode(f1), b.friction[b2], fric_mode(f2));
  e = combine_coeff(b.restitution[b1], rest_mode(f1), b.restitution[b2], rest_mode(f2));
  if (!b.mat_id) return;
  const int i1 = b.mat_id[b1], i2 = b.mat_id[b2];
  if (i1 < 0 || i2 < 0) return;
  const unsigned long long lo = unsigned(i1 < i2 ? i1 : i2), hi = unsigned(i1 < i2 ? i2 : i1);
  const unsigned long long key = (lo << 32) | hi;
  float v;
  if (mat_lookup(mt.fkey, mt.fval, mt.nf, key, v)) mu = v;
  if (mat_lookup(mt.rkey, mt.rval, mt.nr, key, v)) e = v;
}

__global__ void __launch_bounds__(256) k_assemble(DevBodies b, DevContacts cur, DevContacts prev, int prevM,
                                                 int M, SimParams p, SolverBufs sb, MatTable mt) {
  // manifold order (neighbouring lanes read neighbouring bodies and contacts); the records go to
  // the manifold's slot in colour order
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  const uint2 at = sb.slot_of[m];
  const int s = int(at.x);
  const int2 bb = cur.mbody[m];
  const int b1 = bb.x, b2 = bb.y;
  const bool d1 = b.status[b1] == STATUS_DYNAMIC;
  const bool d2 = b.status[b2] == STATUS_DYNAMIC;
  float mu, e;
  material_coefficients(b, mt, b1, b2, mu, e);
  // surface_velocity = position1 * v1 - position2 * v2 (material.rs:175, basic_material.rs:47-56)
  f3 sv{0.0f, 0.0f, 0.0f};
  if (b.surf_vel) sv = sub(qrot(toq(b.rot(b1)), xyz(b.surf_vel[b1])), qrot(toq(b.rot(b2)), xyz(b.surf_vel[b2])));
  const float m1 = b.margin[b1], m2 = b.margin[b2];
  BodyView v1, v2;
  if (d1) v1 = load_body(b, b1);
  if (d2) v2 = load_body(b, b2);
  // previous manifold with the same bodies
  int pf = 0, pc = 0;
  {
    const int j = find_manifold(prev, prevM, b1, b2);
    if (j >= 0) {
      pf = prev.mfirst[j];
      pc = prev.mcount[j];
    }
  }
  const int first = cur.mfirst[m], cnt = cur.mcount[m];
  const uint32_t r0 = at.y;
  // the position solver's inputs in slot / record order (see k_position.hip)
  const int k1 = b.shape[b1], k2 = b.shape[b2];
  sb.pgeo[2 * long(s)] = f4(xyz(b.dims[b1]), m1);
  sb.pgeo[2 * long(s) + 1] = f4(xyz(b.dims[b2]), m2);
  for (int k = 0; k < cnt; ++k) {
    const int c = first + k;
    const uint32_t r = r0 + k;
    const float4* K = cur.contact(c);
    const float4 w14 = K[0], w24 = K[1], n4 = K[2];
    float4* P = sb.prec + 3 * long(r);
    P[0] = f4(xyz(K[3]), n4.w);  // the kinematic kind's bits
    P[1] = f4(xyz(K[4]), __int_as_float(k1));
    P[2] = f4(xyz(K[5]), __int_as_float(k2));
    const f3 n = xyz(n4);
    const f3 w1 = xyz(w14), w2 = xyz(w24);
    const float depth = w14.w;
    const uint32_t feat = __float_as_uint(w24.w);
    float4 imp = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float has = 0.0f;
    for (int kk = 0; kk < pc; ++kk)
      if (prev.feature(pf + kk) == feat) {
        const float4 q = prev.imp[pf + kk];
        if (q.w >= 0.0f) {  // w < 0: a sleeping contact that had no cached impulse
          imp = q;
          has = 1.0f;
        }
        break;
      }
    const f3 center1 = add(w1, scale(n, m1));
    const f3 center2 = sub(w2, scale(n, m2));
    const f3 seed = tangent_seed(n);
    const float tl = sqrtf(dot(seed, seed));
    f3 t1, t2;
    tangents(n, tl, t1, t2);
    float rr3[3], rhs3[3];
    float lam[3];
#pragma unroll
    for (int row = 0; row < 3; ++row) {
      const f3 dir = row == 0 ? neg(n) : (row == 1 ? t1 : t2);
      // n . surface_velocity for the normal row, t . surface_velocity for the friction rows
      float inv_r = 0.0f, rhs = b.surf_vel ? dot(row == 0 ? n : dir, sv) : 0.0f;
      f3 a1{0.0f, 0.0f, 0.0f}, wa1{0.0f, 0.0f, 0.0f}, a2{0.0f, 0.0f, 0.0f}, wa2{0.0f, 0.0f, 0.0f};
      if (d1) fill_geom(v1, center1, dir, a1, wa1, inv_r, rhs);
      if (d2) fill_geom(v2, center2, neg(dir), a2, wa2, inv_r, rhs);
      const float rr = inv_r != 0.0f ? 1.0f / inv_r : 1.0f;
      if (row == 0) {
        if (rhs <= -p.restitution_threshold) rhs = rhs + e * rhs;
        const float de = (depth + m1) + m2;
        if (de < 0.0f) rhs = rhs + (-de) * p.inv_dt;
      }
      rr3[row] = rr;
      rhs3[row] = rhs;
    }
    // lever arms of the contact point from each dynamic body's centre (fill_geom's p); the sweeps
    // rebuild every row's angular jacobian from them with fill_geom's own cross product
    const f3 zero{0.0f, 0.0f, 0.0f};
    const f3 p1 = d1 ? sub(center1, v1.com) : zero;
    const f3 p2 = d2 ? sub(center2, v2.com) : zero;
    lam[0] = imp.x * p.warmstart_coeff;
    lam[1] = imp.y * p.warmstart_coeff;
    lam[2] = imp.z * p.warmstart_coeff;
    float4* R = sb.rec + long(r) * kRecFields;
    R[0] = f4(n, tl);
    R[1] = f4(p1, rr3[0]);
    R[2] = f4(p2, rr3[1]);
    R[3] = make_float4(rhs3[0], rhs3[1], rhs3[2], rr3[2]);
    sb.lam[r] = make_float4(lam[0], lam[1], lam[2], mu);
    if (sb.has) sb.has[r] = has;
  }
}

// Per-lane solver state of one manifold.
struct Dv {
  f3 l, a;
};

__device__ __forceinline__ float dot6(f3 dl, f3 ang, const Dv& v) {
  float s = 0.0f;
  s = s + dl.x * v.l.x;
  s = s + dl.y * v.l.y;
  s = s + dl.z * v.l.z;
  s = s + ang.x * v.a.x;
  s = s + ang.y * v.a.y;
  s = s + ang.z * v.a.z;
  return s;
}

__device__ __forceinline__ void axpy6(float alpha, f3 wl, f3 wa, Dv& v) {
  v.l.x = v.l.x + alpha * wl.x;
  v.l.y = v.l.y + alpha * wl.y;
  v.l.z = v.l.z + alpha * wl.z;
  v.a.x = v.a.x + alpha * wa.x;
  v.a.y = v.a.y + alpha * wa.y;
  v.a.z = v.a.z + alpha * wa.z;
}

struct SlotCtx {
  int b1, b2, cnt, first;
  bool d1, d2;
  uint32_t r0;
};

// One 16-byte load gives everything a lane needs about its manifold (see k_colour_scatter).
__device__ __forceinline__ SlotCtx slot_ctx(const SolverBufs& sb, int s) {
  const int4 q = sb.sinfo[s];
  SlotCtx x;
  x.b1 = q.x & 0x3fffffff;
  x.b2 = q.y & 0x3fffffff;
  x.d1 = (q.x >> 30) & 1;
  x.d2 = (q.y >> 30) & 1;
  x.r0 = uint32_t(q.z);
  x.cnt = q.w & 7;
  x.first = int(uint32_t(q.w) >> 3);
  return x;
}

// A contact's record in registers. The tangents and the inverse-inertia weighted angular
// jacobians are not stored: they are recomputed with the expressions k_assemble evaluates
// (tangents(n) and mulv(I^-1, J_ang)), so they carry the same FP32 values.
struct CRec {
  f3 n;
  float tl, mu;
  f3 p1, p2;  // lever arms (zero for a static body)
  float r[3], rhs[3];
  float4 lam;
};

// Angular jacobians of one row along d (d for body 1, -d for body 2), as fill_geom forms them.
__device__ __forceinline__ f3 ang1(const CRec& c, f3 d) { return cross(c.p1, d); }
__device__ __forceinline__ f3 ang2(const CRec& c, f3 d) { return cross(c.p2, neg(d)); }

__device__ __forceinline__ void load_rec(const SolverBufs& sb, uint32_t r, CRec& c) {
  const float4* p = sb.rec + long(r) * kRecFields;
  const float4 v0 = p[0], v1 = p[1], v2 = p[2], v3 = p[3];
  c.n = xyz(v0);
  c.tl = v0.w;
  c.p1 = xyz(v1);
  c.p2 = xyz(v2);
  c.r[0] = v1.w;
  c.r[1] = v2.w;
  c.r[2] = v3.w;
  c.rhs[0] = v3.x;
  c.rhs[1] = v3.y;
  c.rhs[2] = v3.z;
  c.lam = sb.lam[r];
  c.mu = c.lam.w;
}

// Jacobian masks of a manifold's two bodies (only the masked kernel variants carry them).
template <bool kMask>
struct Masks {
  __device__ void load(const DevBodies&, const SlotCtx&) {}
  __device__ f3 l1(f3 d) const { return d; }
  __device__ f3 l2(f3 d) const { return d; }
  __device__ f3 a1(f3 a) const { return a; }
  __device__ f3 a2(f3 a) const { return a; }
};
template <>
struct Masks<true> {
  f3 ml1, ma1, ml2, ma2;
  __device__ void load(const DevBodies& b, const SlotCtx& x) {
    b.mask(x.b1, ml1, ma1);
    b.mask(x.b2, ml2, ma2);
  }
  __device__ f3 l1(f3 d) const { return cmul(d, ml1); }
  __device__ f3 l2(f3 d) const { return cmul(d, ml2); }
  __device__ f3 a1(f3 a) const { return cmul(a, ma1); }
  __device__ f3 a2(f3 a) const { return cmul(a, ma2); }
};

template <bool kMask>
struct Manifold {
  SlotCtx x;
  CRec c[4];
  f3 t1[4], t2[4];
  Masks<kMask> mk;
};

// A whole manifold on one lane (the residual), loaded up front: all loads are in flight together.
template <bool kMask>
__device__ __forceinline__ void load_manifold(const DevBodies& b, const SolverBufs& sb, int s, Manifold<kMask>& m) {
  m.x = slot_ctx(sb, s);
  m.mk.load(b, m.x);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (k < m.x.cnt) {
      load_rec(sb, m.x.r0 + k, m.c[k]);
      tangents(m.c[k].n, m.c[k].tl, m.t1[k], m.t2[k]);
    }
}

// Row `row` (0 normal, 1 and 2 friction) of contact k, for w = J dv + rhs. Both bodies' terms are always
// evaluated, a static body having a zero dv: its terms are then exact zeros, so w equals the
// one-body expression (up to the sign of a zero), and a wavefront mixing ground and body-body
// manifolds runs one code path. The masked variant multiplies each body's jacobian by its mask,
// as k_assemble's fill_geom does.
struct Row {
  f3 d1, d2, a1, a2;
  float r, rhs;
};

template <bool kMask>
__device__ __forceinline__ Row row_of(const Manifold<kMask>& m, int k, int row) {
  Row v;
  const CRec& c = m.c[k];
  const f3 d = row == 0 ? neg(c.n) : (row == 1 ? m.t1[k] : m.t2[k]);
  v.d1 = m.mk.l1(d);
  v.d2 = m.mk.l2(neg(d));
  v.a1 = m.mk.a1(ang1(c, d));
  v.a2 = m.mk.a2(ang2(c, d));
  v.r = c.r[row];
  v.rhs = c.rhs[row];
  return v;
}

__device__ __forceinline__ float row_w(const Row& v, const Dv& x1, const Dv& x2) {
  return (dot6(v.d1, v.a1, x1) + dot6(v.d2, v.a2, x2)) + v.rhs;
}

template <bool kMask>
__device__ __forceinline__ void load_dv(const DevBodies& b, const Manifold<kMask>& m, Dv& v1, Dv& v2) {
  if (m.x.d1) b.load_dv(m.x.b1, v1.l, v1.a);
  if (m.x.d2) b.load_dv(m.x.b2, v2.l, v2.a);
}

// The value of the other lane of the pair: a quad permutation (1, 0, 3, 2), one instruction, where a
// shuffle goes through the LDS crossbar and stands in every row's serial chain. Both lanes of a pair
// are always active together: they take the same branches, on the same values.
__device__ __forceinline__ float pair_swap(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true));
}

// A contact as one lane of the pair needs it: the normal, the seed's length, its body's lever arm,
// the r of the first two rows (its own record word's and the other's), of the third, the three rhs,
// the impulses and mu. Nothing is computed on loading: a lane that loads ahead must not wait here.
struct CHalf {
  float4 n, p;  // n|length, p|r (row 0 on lane 0, row 1 on lane 1)
  float ro;     // the other of the two
  float4 rhs;   // rhs 0-2|r of row 2
  float4 lam;
  __device__ float r(int row, int h) const { return row == 2 ? rhs.w : ((row == h) ? p.w : ro); }
};

__device__ __forceinline__ void load_half(const SolverBufs& sb, uint32_t r, int h, CHalf& c) {
  const float4* q = sb.rec + long(r) * kRecFields;
  c.n = q[0];
  c.p = q[1 + h];
  c.ro = q[2 - h].w;
  c.rhs = q[3];
  c.lam = sb.lam[r];
}

// One lane's half of a manifold: its body's inverse mass and inertia (zero for a static body), its
// jacobian masks, the contacts. Body 2's jacobians are those of body 1's direction negated, so its
// lane keeps the velocity increment negated instead and both lanes run the same expressions on d:
// (-d).v = d.(-v) and -(v + a (-w)) = -v + a w, the same roundings (up to the sign of a zero).
template <bool kMask>
struct PairHalf {
  int body, cnt, h;
  bool dyn;
  uint32_t r0;
  float im;
  m33 I;
  f3 ml, ma;
  CHalf c[4];
};

template <bool kMask>
__device__ __forceinline__ void load_pair(const DevBodies& b, const SolverBufs& sb, int4 q, int h, PairHalf<kMask>& m) {
  const int w = h ? q.y : q.x;
  m.h = h;
  m.body = w & 0x3fffffff;
  m.dyn = (w >> 30) & 1;
  m.r0 = uint32_t(q.z);
  m.cnt = q.w & 7;
  m.im = 0.0f;
  m.I = m33{};
  if (m.dyn) m.I = load_inv(b, m.body, m.im);
  if (kMask) b.mask(m.body, m.ml, m.ma);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (k < m.cnt) load_half(sb, m.r0 + k, h, m.c[k]);
}

__device__ __forceinline__ void flip(Dv& v) {
  v.l = neg(v.l);
  v.a = neg(v.a);
}

// The velocity increment of the lane's body in memory: zero for a static one.
template <class Lane>
__device__ __forceinline__ void load_pair_dv(const DevBodies& b, const Lane& m, Dv& v) {
  if (!m.dyn) return;
  b.load_dv(m.body, v.l, v.a);
  if (m.h) flip(v);
}

template <class Lane>
__device__ __forceinline__ void store_pair_dv(const DevBodies& b, const Lane& m, Dv& v) {
  if (!m.dyn) return;
  if (m.h) flip(v);
  b.store_dv(m.body, v.l, v.a);
}

// The lane's half of the row along d: the jacobian (masked) and its weighted angular part.
template <bool kMask>
__device__ __forceinline__ void half_row(const PairHalf<kMask>& m, f3 p, f3 d, f3& dh, f3& ah, f3& wah) {
  const f3 a = cross(p, d);
  dh = kMask ? cmul(d, m.ml) : d;
  ah = kMask ? cmul(a, m.ma) : a;
  wah = mulv(m.I, ah);
}

// The tangents of contact c, the seed's quotients one per lane.
__device__ __forceinline__ void pair_tangents(const CHalf& c, int h, f3& t1, f3& t2) {
  const bool sel = fabsf(c.n.x) > fabsf(c.n.y);
  const float a0 = sel ? c.n.z : -c.n.z, a1 = sel ? -c.n.x : c.n.y;
  const float mine = (h ? a1 : a0) / c.n.w, other = pair_swap(mine);
  const float u = h ? other : mine, v = h ? mine : other;
  t2 = sel ? f3{u, 0.0f, v} : f3{0.0f, u, v};
  t1 = cross(t2, xyz(c.n));
}

// Warm start of one manifold (SORProx::warmstart_set, sor_prox.rs:19-45): dv += l W J for every
// row with l != 0, normal rows first, then friction rows. The lanes need nothing of each other but the
// quotients of the tangents; that of a static body runs along for them.
template <bool kMask>
__device__ __forceinline__ void pair_warm(const PairHalf<kMask>& m, Dv& v) {
  f3 dh, ah, wah;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (k >= m.cnt) break;
    if (m.c[k].lam.x == 0.0f) continue;
    half_row(m, xyz(m.c[k].p), neg(xyz(m.c[k].n)), dh, ah, wah);
    axpy6(m.c[k].lam.x, scale(dh, m.im), wah, v);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (k >= m.cnt) break;
    if (m.c[k].lam.y == 0.0f && m.c[k].lam.z == 0.0f) continue;
    f3 t1, t2;
    pair_tangents(m.c[k], m.h, t1, t2);
    if (m.c[k].lam.y != 0.0f) {
      half_row(m, xyz(m.c[k].p), t1, dh, ah, wah);
      axpy6(m.c[k].lam.y, scale(dh, m.im), wah, v);
    }
    if (m.c[k].lam.z != 0.0f) {
      half_row(m, xyz(m.c[k].p), t2, dh, ah, wah);
      axpy6(m.c[k].lam.z, scale(dh, m.im), wah, v);
    }
  }
}

// One lane of a contact of a manifold: its body's inverse mass and inertia and jacobian masks, the contact.
// The loads are unconditional, so that none waits for a branch: a static body's solver block
// holds zeros, and a lane without a contact of its own (k >= cnt) reads the manifold's last one.
template <bool kMask>
struct ContactLane {
  int body, cnt, k, h;
  bool dyn;
  uint32_t r;  // its record
  float4 i0, i1, i2;
  f3 ml, ma;
  CHalf c;
};

template <bool kMask>
__device__ __forceinline__ void load_lane(const DevBodies& b, const SolverBufs& sb, int4 q, int k, int h,
                                          ContactLane<kMask>& m) {
  const int w = h ? q.y : q.x;
  m.k = k;
  m.h = h;
  m.body = w & 0x3fffffff;
  m.dyn = (w >> 30) & 1;
  m.cnt = q.w & 7;
  m.r = uint32_t(q.z) + uint32_t(k < m.cnt ? k : (m.cnt > 0 ? m.cnt - 1 : 0));
  const float4* s = b.solver(m.body);
  m.i0 = s[0];
  m.i1 = s[1];
  m.i2 = s[2];
  load_half(sb, m.r, h, m.c);
  if (kMask) b.mask(m.body, m.ml, m.ma);
}

// The value two lanes before, within the sixteen lanes of a row: the pair of the previous contact.
__device__ __forceinline__ float pair_before(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x112, 0xf, 0xf, true));
}

// One SOR-Prox step of a manifold (sor_prox.rs:159-343) on its lanes, contact by contact: the normal
// row, projected on l >= 0, then the two friction rows, bounded by mu times that normal impulse
// and zeroed when it is zero. Both lanes of a pair form w = (s1 + s2) + rhs and the same new impulse.
// v enters on the first pair of lanes and leaves on the last contact's. What the rows are made of does
// not depend on v and is formed for all contacts at once; the wave takes as many turns as its largest manifold.
template <bool kMask>
__device__ __forceinline__ void sweep_lanes(ContactLane<kMask>& m, Dv& v) {
  CHalf& c = m.c;
  m33 I;
  I.m[0][0] = m.i0.x; I.m[0][1] = m.i0.y; I.m[0][2] = m.i0.z;
  I.m[1][0] = m.i1.x; I.m[1][1] = m.i1.y; I.m[1][2] = m.i1.z;
  I.m[2][0] = m.i1.w; I.m[2][1] = m.i2.x; I.m[2][2] = m.i2.y;
  const float im = m.i0.w;
  f3 d[3], a[3], wl[3], wa[3];
  d[0] = neg(xyz(c.n));
  pair_tangents(c, m.h, d[1], d[2]);
#pragma unroll
  for (int row = 0; row < 3; ++row) {
    a[row] = cross(xyz(c.p), d[row]);
    if (kMask) {
      d[row] = cmul(d[row], m.ml);
      a[row] = cmul(a[row], m.ma);
    }
    wl[row] = scale(d[row], im);
    wa[row] = mulv(I, a[row]);
  }
  for (int turn = 0;;) {
    if (m.k == turn && turn < m.cnt) {
      {
        const float s = dot6(d[0], a[0], v);
        const float w = (s + pair_swap(s)) + c.rhs.x;
        const float x = c.lam.x - c.r(0, m.h) * w;
        const float ni = x > 0.0f ? x : 0.0f;
        const float dl = ni - c.lam.x;
        c.lam.x = ni;
        axpy6(dl, wl[0], wa[0], v);
      }
      const float ln = c.lam.x;
#pragma unroll
      for (int f = 1; f <= 2; ++f) {
        float li = f == 1 ? c.lam.y : c.lam.z;
        if (ln == 0.0f) {
          if (li != 0.0f) {
            axpy6(-li, wl[f], wa[f], v);
            li = 0.0f;
          }
        } else {
          const float mx = c.lam.w * ln;
          const float mn = -mx;
          const float s = dot6(d[f], a[f], v);
          const float w = (s + pair_swap(s)) + (f == 1 ? c.rhs.y : c.rhs.z);
          const float val = li - c.r(f, m.h) * w;
          const float ni = val > mn ? (val < mx ? val : mx) : mn;
          const float dl = ni - li;
          li = ni;
          axpy6(dl, wl[f], wa[f], v);
        }
        if (f == 1) c.lam.y = li;
        else c.lam.z = li;
      }
    }
    ++turn;
    if (!__any(m.cnt > turn)) break;
    const Dv u{f3{pair_before(v.l.x), pair_before(v.l.y), pair_before(v.l.z)},
               f3{pair_before(v.a.x), pair_before(v.a.y), pair_before(v.a.z)}};
    if (m.k == turn) v = u;
  }
}

// Whether this lane's pair holds the manifold's result.
template <bool kMask>
__device__ __forceinline__ bool last_pair(const ContactLane<kMask>& m) {
  return m.dyn && m.k == m.cnt - 1;
}

template <bool kMask>
__device__ __forceinline__ void store_lane_lam(const SolverBufs& sb, const ContactLane<kMask>& m) {
  if (m.h == 0 && m.k < m.cnt) sb.lam[m.r] = m.c.lam;
}

// Slot and contact of lane L of a class, or false beyond its lanes.
__device__ __forceinline__ bool lane_at(const ClassSpan& c, int L, int& slot, int& k) {
  const bool several = L < 8 * c.multi;
  const int l = L - 8 * c.multi;
  slot = several ? c.first + (L >> 3) : c.first + c.multi + (l >> 1);
  k = several ? (L >> 1) & 3 : 0;
  return several || l < 2 * c.single;
}

// Lane L's part of the warm start of a class (two lanes per manifold) or of one sweep, at velocity increments in memory.
template <bool kWarm, bool kMask>
__device__ __forceinline__ void class_lane(const DevBodies& b, const SolverBufs& sb, const ClassSpan& c, int L) {
  Dv v{};
  if (kWarm) {
    if ((L >> 1) >= c.multi + c.single) return;
    PairHalf<kMask> m;
    load_pair(b, sb, sb.sinfo[c.first + (L >> 1)], L & 1, m);
    load_pair_dv(b, m, v);
    pair_warm(m, v);
    store_pair_dv(b, m, v);
  } else {
    int slot, k;
    if (!lane_at(c, L, slot, k)) return;
    ContactLane<kMask> m;
    load_lane(b, sb, sb.sinfo[slot], k, L & 1, m);
    load_pair_dv(b, m, v);
    sweep_lanes(m, v);
    if (last_pair(m)) store_pair_dv(b, m, v);
    store_lane_lam(sb, m);
  }
}

// One colour of the warm start or of one sweep. A launch's latency bounds it: ids, then body and
// contact, then the manifold's contacts in turn. With the contacts of a manifold in a loop on two lanes
// the rows of each were formed in its turn; on lanes of their own they are formed at once:
// velocity solve 460 -> 412 us at 10,795 manifolds of 3.3 contacts, 1,554 -> 1,439 at 248,353 of 1.3.
template <bool kWarm, bool kMask>
__global__ void __launch_bounds__(64) k_pgs(DevBodies b, SolverBufs sb, ClassSpan c) {
  class_lane<kWarm, kMask>(b, sb, c, blockIdx.x * 64 + threadIdx.x);
}

// A run of consecutive small colour classes of the visiting order in one workgroup, a barrier
// between classes: per body the same updates in the same order as one launch per class, without
// a launch per class. Each class fits one pass of the workgroup, whose compute unit's issue rate bounds it
// (the next class's ids loaded ahead: no gain).
template <bool kWarm, bool kMask>
__global__ void __launch_bounds__(kRunLanes) k_colour_run(DevBodies b, SolverBufs sb, ClassRun run) {
  for (int k = 0; k < run.n; ++k) {
    class_lane<kWarm, kMask>(b, sb, run.r[k], threadIdx.x);
    __syncthreads();
  }
}

// Scene-blocked sweeps: one workgroup per scene runs the warm start (when warm) and nsweeps sweeps over
// all colours in the visiting order, on the lanes that k_pgs gives a class, the scene's dynamic-body velocity increments
// resident in LDS and a barrier between colours. Every body sees the same sequence of row updates as
// under the per-colour launches (manifolds of one colour share no dynamic body; colours and sweeps
// keep their order), so the results are identical.
//
// A phase (one colour) is short, so what it waits for decides: the body and the contact of a
// lane's next phase are loaded while this one is solved, and the ids of the one after (info, in the scene's
// order). No load's latency stands between two barriers, and the barrier orders LDS alone. Impulses are stored before
// the barrier and read again visit.n - 1 phases later at the earliest (visit.n >= 2): the stores of
// all earlier phases are waited for before a phase's loads are issued. With 1,024 lanes (128 registers each) a second
// contact in flight would spill, and four waves per SIMD cover its loads: sweeps 493 -> 426 us in a pile of 1,900
// without it, 608 -> 461 with jacobian masks (512 lanes: 557 and 593). The scene's one compute unit
// bounds it, by its issue rate: 428 us at 1,021 scenes of 100 bodies (405 with a launch per class),
// 188 against 155 at one of 1,001, and faster where many tiny classes follow one another.
struct SceneItem {
  int4 q;
  int k, local;  // contact, rank of this lane's body in its scene (static: any)
};

__device__ __forceinline__ void barrier_lds() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int kBlock, int kCap, bool kMask>
__global__ void __launch_bounds__(kBlock) k_sweeps_blocked(DevBodies b, SolverBufs sb, SceneBlocks sc,
                                                         const int* __restrict__ scene_list, VisitOrder visit,
                                                         int nsweeps, int warm) {
  __shared__ float4 s_a[kCap];  // linear x, y, z, angular x
  __shared__ float2 s_b[kCap];  // angular y, z
  __shared__ ClassSpan s_span[kVisitColours];
  constexpr bool kAhead = kBlock <= 512;
  const int s = scene_list[blockIdx.x], tid = threadIdx.x, h = tid & 1;
  const int d0 = sc.dyn_start[s], nd = sc.dyn_start[s + 1] - d0;
  const int n = visit.n;
  for (int k = tid; k < n; k += kBlock) s_span[k] = scene_span(sc, visit, s, k);
  for (int i = tid; i < nd; i += kBlock) {
    f3 l, a;
    b.load_dv(sc.dyn_list[d0 + i], l, a);
    s_a[i] = make_float4(l.x, l.y, l.z, a.x);
    s_b[i] = make_float2(a.y, a.z);
  }
  __syncthreads();
  auto item = [&](int class_at, int L, SceneItem& it) {
    int at;
    it.q = make_int4(0, 0, 0, 0);  // a manifold without contacts
    it.local = 0;
    const bool in = lane_at(s_span[class_at], L, at, it.k);
    if (in) {
      it.q = sc.info[at];
      it.local = reinterpret_cast<const int*>(sc.rank)[2 * at + h];
    }
    return in;
  };
  auto load_v = [&](bool dyn, int local, Dv& v) {
    v = Dv{};
    if (!dyn) return;
    const float4 x = s_a[local];
    const float2 y = s_b[local];
    v.l = xyz(x);
    v.a = f3{x.w, y.x, y.y};
    if (h) flip(v);
  };
  auto store_v = [&](int local, Dv& v) {
    if (h) flip(v);
    s_a[local] = make_float4(v.l.x, v.l.y, v.l.z, v.a.x);
    s_b[local] = make_float2(v.a.y, v.a.z);
  };
  if (warm) {
    for (int k = 0; k < n; ++k) {
      const ClassSpan c = s_span[k];
      for (int t = tid; (t >> 1) < c.multi + c.single; t += kBlock) {
        PairHalf<kMask> m;
        const int at = c.first + (t >> 1);
        load_pair(b, sb, sc.info[at], h, m);
        const int local = reinterpret_cast<const int*>(sc.rank)[2 * at + h];
        Dv v;
        load_v(m.dyn, local, v);
        pair_warm(m, v);
        if (m.dyn) store_v(local, v);
      }
      barrier_lds();
    }
  }
  auto after = [&](int c) { return c + 1 < n ? c + 1 : 0; };
  int k = 0;  // class visited in this phase
  SceneItem it, here;
  ContactLane<kMask> next;
  item(0, tid, here);
  if (kAhead) load_lane(b, sb, here.q, here.k, h, next);
  item(after(0), tid, it);
  for (int ph = 0; ph < n * nsweeps; ++ph) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    ContactLane<kMask> m;
    if (kAhead) m = next;
    else load_lane(b, sb, here.q, here.k, h, m);
    int local = here.local;
    here = it;
    if (kAhead) load_lane(b, sb, it.q, it.k, h, next);
    item(after(after(k)), tid, it);
    for (int L = tid;;) {
      if (m.cnt) {
        Dv v;
        load_v(m.dyn, local, v);
        sweep_lanes(m, v);
        if (last_pair(m)) store_v(local, v);
        store_lane_lam(sb, m);
      }
      L += kBlock;  // the class's manifolds beyond one workgroup's worth
      SceneItem more;
      if (!item(k, L, more)) break;
      load_lane(b, sb, more.q, more.k, h, m);
      local = more.local;
    }
    barrier_lds();
    k = after(k);
  }
  for (int i = tid; i < nd; i += kBlock) {
    const float4 x = s_a[i];
    const float2 y = s_b[i];
    b.store_dv(sc.dyn_list[d0 + i], xyz(x), f3{x.w, y.x, y.y});
  }
}

// Scene-major slot order for the blocked kernels: the slots are in colour order, so a stable sort by scene
// leaves them in (scene, colour) order.
__global__ void __launch_bounds__(256) k_scene_keys(DevBodies b, int M, SolverBufs sb, uint32_t* keys,
                                                   uint32_t* slots) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  const int b1 = sb.sinfo[i].x & 0x3fffffff;
  keys[i] = uint32_t(b.scene[b1]);
  slots[i] = uint32_t(i);
}

// The slots' records in that order (one scene: in slot order), each with its bodies' ranks in their scene.
__global__ void __launch_bounds__(256) k_scene_info(int M, SolverBufs sb, SceneBlocks sc) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  const int4 q = sb.sinfo[sc.at(i)];
  sc.info[i] = q;
  sc.rank[i] = make_int2(sc.local[q.x & 0x3fffffff], sc.local[q.y & 0x3fffffff]);
}

// start[s][d] = first position of (scene s, digit of the colour order >= d) in the sorted slots (lower bound).
__global__ void __launch_bounds__(256) k_scene_starts(const uint32_t* __restrict__ keys,
                                                     const uint32_t* __restrict__ slot,
                                                     const uint32_t* __restrict__ colour, int M, int nscenes,
                                                     int ncolours, uint32_t* start) {
  const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
  const long total = long(nscenes) * (ncolours + 1);
  if (t >= total) return;
  const int s = int(t / (ncolours + 1)), c = int(t % (ncolours + 1));
  int lo = 0, hi = M;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    const int ks = int(keys[mid]);
    if (ks < s || (ks == s && int(colour[slot[mid]]) < c)) lo = mid + 1;
    else hi = mid;
  }
  start[t] = uint32_t(lo);
}

// What the next step's assembly finds of a solved contact (w >= 0: there is a cached impulse).
__device__ __forceinline__ float4 cached_impulse(float4 lam) { return make_float4(lam.x, lam.y, lam.z, 0.0f); }

// Natural-map residual per row; per block (max |phi|, sum phi^2) in double, written to host memory and
// reduced there in block order. With kCache the manifold's impulses, which it has in registers, go to
// the contacts' slots as well (cache_impulses: the warm start of the next step), 16 to 64 contiguous bytes.
// No fence to the host here: the readback kernel behind it on the stream releases at system scope, for all that
// happened before it. One per workgroup wrote the L2 back, impulses and all, each time: 258 -> 73 us at 1,145,425 manifolds (89
// with the impulses in a kernel of their own and the partials in device memory), 136 -> 42 at 503,230.
template <bool kMask, bool kCache>
__global__ void __launch_bounds__(256) k_residual(DevBodies b, DevContacts c, int M, SolverBufs sb) {
  __shared__ double s_max[256];
  __shared__ double s_sum[256];
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  double mx = 0.0, sum = 0.0;
  if (s < M) {
    Manifold<kMask> m;
    load_manifold(b, sb, s, m);
    Dv v1{}, v2{};
    load_dv(b, m, v1, v2);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k >= m.x.cnt) break;
      const float4 lam = m.c[k].lam;
      if (kCache) c.imp[m.x.first + k] = cached_impulse(lam);
      {
        const Row v = row_of(m, k, 0);
        const float w = row_w(v, v1, v2);
        const float a = lam.x - v.r * w;
        const float pr = a > 0.0f ? a : 0.0f;
        const double phi = fabs(double((lam.x - pr) / v.r));
        mx = phi > mx ? phi : mx;
        sum += phi * phi;
      }
#pragma unroll
      for (int f = 1; f <= 2; ++f) {
        const float li = f == 1 ? lam.y : lam.z;
        const Row v = row_of(m, k, f);
        const float w = row_w(v, v1, v2);
        const float mxv = m.c[k].mu * lam.x, mnv = -mxv;
        const float val = li - v.r * w;
        const float pr = val > mnv ? (val < mxv ? val : mxv) : mnv;
        const double phi = fabs(double((li - pr) / v.r));
        mx = phi > mx ? phi : mx;
        sum += phi * phi;
      }
    }
  }
  s_max[threadIdx.x] = mx;
  s_sum[threadIdx.x] = sum;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      s_max[threadIdx.x] = s_max[threadIdx.x] > s_max[threadIdx.x + off] ? s_max[threadIdx.x] : s_max[threadIdx.x + off];
      s_sum[threadIdx.x] += s_sum[threadIdx.x + off];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    sb.red[2 * blockIdx.x] = s_max[0];
    sb.red[2 * blockIdx.x + 1] = s_sum[0];
  }
}

__global__ void __launch_bounds__(256) k_cache(DevContacts c, int M, SolverBufs sb) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= M) return;
  const SlotCtx x = slot_ctx(sb, s);
  for (int k = 0; k < x.cnt; ++k) c.imp[x.first + k] = cached_impulse(sb.lam[x.r0 + k]);
}

// ------------------------------------------------------------------ learned warm start
// Features of every contact row record (the network's 24 inputs, in the order documented with
// nphys_mlp_create), computed after assembly from the record, the bodies and the contact:
// velocities over |g| dt, depth over |g| dt^2, mass terms over the row's inverse effective mass,
// cached impulses over ls = r_n |g| dt (the impulse that cancels |g| dt along the normal), which
// is also written per record as the network's output unit.
__global__ void __launch_bounds__(256) k_features(DevBodies b, DevContacts cur, SimParams p, int M, SolverBufs sb,
                                                  float* __restrict__ X, float* __restrict__ ls) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= M) return;
  const SlotCtx x = slot_ctx(sb, s);
  float im1 = 0.0f, im2 = 0.0f;
  m33 I1, I2;
  if (x.d1) I1 = load_inv(b, x.b1, im1);
  if (x.d2) I2 = load_inv(b, x.b2, im2);
  const float g = sqrtf(p.gx * p.gx + p.gy * p.gy + p.gz * p.gz);
  const float gdt = (g > 0.0f ? g : 1.0f) * p.dt;
  const float e = (b.restitution[x.b1] + b.restitution[x.b2]) * 0.5f;
  const float mm = b.margin[x.b1] + b.margin[x.b2];
  for (int k = 0; k < x.cnt; ++k) {
    const uint32_t r = x.r0 + k;
    CRec c;
    load_rec(sb, r, c);
    f3 t1, t2;
    tangents(c.n, c.tl, t1, t2);
    const float depth = cur.contact(x.first + k)[0].w + mm;
    const float lsc = c.r[0] * gdt;
    float* f = X + long(r) * 24;
#pragma unroll
    for (int row = 0; row < 3; ++row) {
      f[row] = c.rhs[row] / gdt;
      const f3 d = row == 0 ? neg(c.n) : (row == 1 ? t1 : t2);
      const f3 j1 = ang1(c, d), j2 = ang2(c, d);
      const float a1 = x.d1 ? dot(j1, mulv(I1, j1)) : 0.0f;
      const float a2 = x.d2 ? dot(j2, mulv(I2, j2)) : 0.0f;
      f[9 + row] = a1 * c.r[row];
      f[12 + row] = a2 * c.r[row];
    }
    f[3] = c.n.x;
    f[4] = c.n.y;
    f[5] = c.n.z;
    f[6] = depth / (gdt * p.dt);
    f[7] = im1 * c.r[0];
    f[8] = im2 * c.r[0];
    f[15] = float(x.cnt) * 0.25f;
    f[16] = c.lam.x / lsc;
    f[17] = c.lam.y / lsc;
    f[18] = c.lam.z / lsc;
    f[19] = c.mu;
    f[20] = e;
    f[21] = gdt;
    f[22] = (x.d1 && x.d2) ? 0.0f : 1.0f;
    f[23] = sb.has[r];
    ls[r] = lsc;
  }
}

// The network predicts the correction of the cache warm start in units of ls: the warm start
// becomes cache + y ls (cache 0 for a new contact), projected on the admissible set (normal >= 0,
// each tangent within +-mu normal, the pyramid of the friction rows).
__global__ void __launch_bounds__(256) k_apply_prediction(SolverBufs sb, int C, const float* __restrict__ y,
                                                          const float* __restrict__ ls) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= C) return;
  const float s = ls[r];
  float4* L = sb.lam + r;
  const float4 c = *L;
  const float mu = c.w;
  const float ln = fmaxf(c.x + y[3 * r] * s, 0.0f);
  const float lim = mu * ln;
  const float t1 = fminf(fmaxf(c.y + y[3 * r + 1] * s, -lim), lim);
  const float t2 = fminf(fmaxf(c.z + y[3 * r + 2] * s, -lim), lim);
  *L = make_float4(ln, t1, t2, c.w);
}

// Training targets of the last solve: the impulses in units of ls.
__global__ void __launch_bounds__(256) k_sample_targets(SolverBufs sb, int C, const float* __restrict__ ls,
                                                        float* __restrict__ t) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= C) return;
  const float4 l = sb.lam[r];
  const float s = ls[r];
  t[3 * r] = l.x / s;
  t[3 * r + 1] = l.y / s;
  t[3 * r + 2] = l.z / s;
}

// Impulses of all records to / from a side buffer (the judge's saved solves).
__global__ void __launch_bounds__(256) k_lam_copy(SolverBufs sb, int C, float4* __restrict__ buf, int to_buf) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= C) return;
  float4* L = sb.lam + r;
  if (to_buf) buf[r] = *L;
  else *L = buf[r];
}

inline unsigned nb(long n) { return unsigned((n + 255) / 256); }

}  // namespace

void launch_colour_begin(const DevBodies& b, const DevContacts& c, int M, const DevContacts& prev, int prevM,
                         const uint32_t* prev_state, SolverBufs& sb, hipStream_t s) {
  fill_u32(sb.deg, 0u, size_t(b.n), s);
  hipLaunchKernelGGL(k_colour_begin, dim3(nb(M)), dim3(256), 0, s, b, c, M, prev, prevM, prev_state, sb);
  scan_exclusive_u32(sb.deg, sb.adj_off, b.n, *sb.scan, s);
  hipLaunchKernelGGL(k_adjacency, dim3(nb(M)), dim3(256), 0, s, c, M, sb);
}

void launch_colour_small(const DevBodies& b, const DevContacts& c, int M, int C, const DevContacts& prev, int prevM,
                         const uint32_t* prev_state, bool split, SolverBufs& sb, uint32_t* words, hipStream_t s) {
  if (split)
    hipLaunchKernelGGL(k_colour_small<true>, dim3(1), dim3(kSmallThreads), 0, s, b, c, M, C, prev, prevM, prev_state, sb,
                       words);
  else
    hipLaunchKernelGGL(k_colour_small<false>, dim3(1), dim3(kSmallThreads), 0, s, b, c, M, C, prev, prevM, prev_state, sb,
                       words);
}

void launch_colour_round(const DevContacts& c, int M, int round, uint32_t* remaining, uint32_t* last_round,
                         SolverBufs& sb, hipStream_t s) {
  // Sixteen lanes up to the manifolds for which that still leaves the chip half empty: then the longest list of
  // neighbours sets the time: 13.9 -> 4.0 us a round at some 2,000 manifolds of a fast crowd. Beyond, most manifolds
  // are coloured already and the lanes would only read that.
  if (M <= 16384)
    hipLaunchKernelGGL(k_colour_round<16>, dim3(nb(16l * M)), dim3(256), 0, s, c, M, uint32_t(round), sb.adj_off,
                       sb.deg, sb.adj, sb.place, sb.state, remaining, last_round);
  else
    hipLaunchKernelGGL(k_colour_round<1>, dim3(nb(M)), dim3(256), 0, s, c, M, uint32_t(round), sb.adj_off, sb.deg,
                       sb.adj, sb.place, sb.state, remaining, last_round);
}

namespace {
template <int kDigits, int kThreads, bool kSplit>
void colour_order(const DevContacts& c, int M, int C, SolverBufs& sb, uint32_t* ncol, hipStream_t s) {
  const int ntiles = (M + kColourTile - 1) / kColourTile;
  hipLaunchKernelGGL((k_colour_hist<kDigits, kThreads, kSplit>), dim3(ntiles), dim3(kThreads), 0, s, c, M, ntiles, sb, ncol);
  scan_exclusive_u32(sb.hist, sb.offs, 2 * kDigits * ntiles, *sb.scan, s);
  hipLaunchKernelGGL((k_colour_scatter<kDigits, kThreads, kSplit>), dim3(ntiles), dim3(kThreads), 0, s, c, M, C, ntiles, sb);
}
}  // namespace

size_t colour_hist_words(int M, int digits) {
  return 2 * size_t(digits) * size_t((M + kColourTile - 1) / kColourTile);
}

void launch_colour_order(const DevContacts& c, int M, int C, int digits, bool split, SolverBufs& sb, uint32_t* ncol,
                         hipStream_t s) {
  if (digits != kColourDigits) colour_order<kMaxColours, 64, false>(c, M, C, sb, ncol, s);
  else if (split) colour_order<kColourDigits, 256, true>(c, M, C, sb, ncol, s);
  else colour_order<kColourDigits, 256, false>(c, M, C, sb, ncol, s);
}

void launch_assemble(const DevBodies& b, const DevContacts& cur, const DevContacts& prev, int prevM,
                     int M, const SimParams& p, SolverBufs& sb, const MatTable& mt, hipStream_t s) {
  if (M == 0) return;
  hipLaunchKernelGGL(k_assemble, dim3(nb(M)), dim3(256), 0, s, b, cur, prev, prevM, M, p, sb, mt);
}

// 64-lane workgroups for a class's lanes (at most 8 a manifold: the grid stays within its limits).
static unsigned lane_blocks(long lanes) { return unsigned(std::max((lanes + 63) / 64, 1l)); }

// The masked kernel variants run only in worlds where some dynamic body has a kinematic dof.
void launch_warmstart_colour(const DevBodies& b, const ClassSpan& c, SolverBufs& sb, hipStream_t s) {
  const dim3 grid(lane_blocks(2l * (c.multi + c.single)));
  if (b.kmask) hipLaunchKernelGGL((k_pgs<true, true>), grid, dim3(64), 0, s, b, sb, c);
  else hipLaunchKernelGGL((k_pgs<true, false>), grid, dim3(64), 0, s, b, sb, c);
}

void launch_pgs_colour(const DevBodies& b, const ClassSpan& c, SolverBufs& sb, hipStream_t s, hipEvent_t ev0,
                       hipEvent_t ev1) {
  const dim3 grid(lane_blocks(8l * c.multi + 2l * c.single));
  // with events, the dispatch packet itself records both, timing the kernel alone
  if (b.kmask) {
    if (ev0) hipExtLaunchKernelGGL((k_pgs<false, true>), grid, dim3(64), 0, s, ev0, ev1, 0, b, sb, c);
    else hipLaunchKernelGGL((k_pgs<false, true>), grid, dim3(64), 0, s, b, sb, c);
    return;
  }
  if (ev0) hipExtLaunchKernelGGL((k_pgs<false, false>), grid, dim3(64), 0, s, ev0, ev1, 0, b, sb, c);
  else hipLaunchKernelGGL((k_pgs<false, false>), grid, dim3(64), 0, s, b, sb, c);
}

void launch_colour_run(const DevBodies& b, SolverBufs& sb, const ClassRun& run, bool warm, hipStream_t s) {
  // as many lanes as the largest class takes: fewer waves meet at each barrier
  int lanes = 64;
  for (int k = 0; k < run.n; ++k) {
    const ClassSpan& c = run.r[k];
    lanes = std::max(lanes, warm ? 2 * (c.multi + c.single) : 8 * c.multi + 2 * c.single);
  }
  const dim3 block(unsigned(std::min((lanes + 63) & ~63, kRunLanes)));
  if (b.kmask) {
    if (warm) hipLaunchKernelGGL((k_colour_run<true, true>), dim3(1), block, 0, s, b, sb, run);
    else hipLaunchKernelGGL((k_colour_run<false, true>), dim3(1), block, 0, s, b, sb, run);
    return;
  }
  if (warm) hipLaunchKernelGGL((k_colour_run<true, false>), dim3(1), block, 0, s, b, sb, run);
  else hipLaunchKernelGGL((k_colour_run<false, false>), dim3(1), block, 0, s, b, sb, run);
}

int residual_blocks(int M) { return int(nb(M > 0 ? M : 1)); }

void launch_residual(const DevBodies& b, const DevContacts& c, int M, bool cache, SolverBufs& sb, hipStream_t s) {
  const dim3 grid(nb(M > 0 ? M : 1));
  if (b.kmask) {
    if (cache) hipLaunchKernelGGL((k_residual<true, true>), grid, dim3(256), 0, s, b, c, M, sb);
    else hipLaunchKernelGGL((k_residual<true, false>), grid, dim3(256), 0, s, b, c, M, sb);
  } else {
    if (cache) hipLaunchKernelGGL((k_residual<false, true>), grid, dim3(256), 0, s, b, c, M, sb);
    else hipLaunchKernelGGL((k_residual<false, false>), grid, dim3(256), 0, s, b, c, M, sb);
  }
}

void launch_cache_impulses(const DevContacts& c, SolverBufs& sb, int M, hipStream_t s) {
  if (M == 0) return;
  hipLaunchKernelGGL(k_cache, dim3(nb(M)), dim3(256), 0, s, c, M, sb);
}

void launch_features(const DevBodies& b, const DevContacts& c, const SimParams& p, int M, SolverBufs& sb, float* X,
                     float* ls, hipStream_t s) {
  if (M == 0) return;
  hipLaunchKernelGGL(k_features, dim3(nb(M)), dim3(256), 0, s, b, c, p, M, sb, X, ls);
}

void launch_apply_prediction(SolverBufs& sb, int C, const float* y, const float* ls, hipStream_t s) {
  if (C == 0) return;
  hipLaunchKernelGGL(k_apply_prediction, dim3(nb(C)), dim3(256), 0, s, sb, C, y, ls);
}

void launch_sample_targets(SolverBufs& sb, int C, const float* ls, float* t, hipStream_t s) {
  if (C == 0) return;
  hipLaunchKernelGGL(k_sample_targets, dim3(nb(C)), dim3(256), 0, s, sb, C, ls, t);
}

void launch_lam_copy(SolverBufs& sb, int C, float4* buf, bool to_buf, hipStream_t s) {
  if (C == 0) return;
  hipLaunchKernelGGL(k_lam_copy, dim3(nb(C)), dim3(256), 0, s, sb, C, buf, to_buf ? 1 : 0);
}

void launch_scene_order(const DevBodies& b, int M, int nscenes, int scene_bits, int digits, SolverBufs& sb,
                        SceneBlocks& sc, hipStream_t s) {
  if (M == 0) return;
  if (sc.slot) {
    hipLaunchKernelGGL(k_scene_keys, dim3(nb(M)), dim3(256), 0, s, b, M, sb, sc.keys, sc.slot);
    radix_sort_pairs(sc.keys, sc.slot, sc.keys_alt, sc.slot_alt, M, (scene_bits + 15) / 16 * 16, sb.tmp, *sb.scan, s);
    const long total = long(nscenes) * (digits + 1);
    hipLaunchKernelGGL(k_scene_starts, dim3(nb(total)), dim3(256), 0, s, sc.keys, sc.slot, sb.ckeys, M, nscenes, digits,
                       sc.start);
  }
  hipLaunchKernelGGL(k_scene_info, dim3(nb(M)), dim3(256), 0, s, M, sb, sc);
}

// Two launches: the scenes with more than kSmallScene dynamic bodies (256, 512 or 1,024 lanes, 54 KB of LDS)
// on s_large, the others (128-lane workgroups, many resident per CU) on s_small, so the few large
// scenes run beside the many small ones.
template <bool kMask>
void sweeps_blocked(const DevBodies& b, SolverBufs& sb, const SceneBlocks& sc, const VisitOrder& visit, int nsweeps,
                    bool warm, int block, hipStream_t s_small, hipStream_t s_large) {
  const int w = warm ? 1 : 0;
  if (sc.n_large > 0) {
    if (block == 256)
      hipLaunchKernelGGL((k_sweeps_blocked<256, kLdsBodies, kMask>), dim3(sc.n_large), dim3(256), 0, s_large, b, sb,
                         sc, sc.large_list, visit, nsweeps, w);
    else if (block == 1024)
      hipLaunchKernelGGL((k_sweeps_blocked<1024, kLdsBodies, kMask>), dim3(sc.n_large), dim3(1024), 0, s_large, b, sb,
                         sc, sc.large_list, visit, nsweeps, w);
    else
      hipLaunchKernelGGL((k_sweeps_blocked<512, kLdsBodies, kMask>), dim3(sc.n_large), dim3(512), 0, s_large, b, sb,
                         sc, sc.large_list, visit, nsweeps, w);
  }
  if (sc.n_small > 0)
    hipLaunchKernelGGL((k_sweeps_blocked<kSmallLanes, kSmallScene, kMask>), dim3(sc.n_small), dim3(kSmallLanes), 0, s_small, b, sb, sc,
                       sc.small_list, visit, nsweeps, w);
}

void launch_sweeps_blocked(const DevBodies& b, SolverBufs& sb, const SceneBlocks& sc, const VisitOrder& visit,
                           int nsweeps, bool warm, int block, hipStream_t s_small, hipStream_t s_large) {
  if (b.kmask) sweeps_blocked<true>(b, sb, sc, visit, nsweeps, warm, block, s_small, s_large);
  else sweeps_blocked<false>(b, sb, sc, visit, nsweeps, warm, block, s_small, s_large);
}

}  // namespace nph
