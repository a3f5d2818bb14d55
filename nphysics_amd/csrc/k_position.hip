// nphysics_amd/csrc/k_position.hip -- coloured nonlinear position correction.
//
// Restates NonlinearSORProx::solve / solve_unilateral / update_contact_constraint / clamp_rhs
// (src/solver/nonlinear_sor_prox.rs:17-55, 121-309): per contact, re-evaluate the contact at the
// current poses (the kinematic of the narrow phase, np_geometry.hpp::reevaluate), dilate by both
// margins (src/solver/signorini_model.rs:174-181), rhs = max((-depth + allowed_linear_error) erp,
// -max_linear_correction); if rhs < 0 move each dynamic body by its weighted jacobian times
// -rhs / (J M^-1 J^T) (RigidBody::apply_displacement, src/object/rigid_body.rs:371-381),
// immediately, so later contacts see the corrected poses.
//
// A manifold has four adjacent lanes, one per contact (position_lanes). All contacts are evaluated at once;
// the first that needs a correction is applied and those after it are evaluated again at the poses
// it leaves, so every contact that moves a body is evaluated at the same poses as one after another,
// but the rounds are as many as there are corrections plus one, not one per contact, and a wavefront runs the code
// of each kind of contact once per round. One lane per manifold took 15 us a launch at 1,200 manifolds
// of cuboids, bound by that chain on a handful of wavefronts; it takes 8 us now, of which launch, loads and one round are 5.
//
// Its inputs are laid out by the assembly in colour order: per slot the two bodies' half extents and
// margins, per contact a 48-byte position record (local points and normal, contact kind, shape
// kinds), so a manifold reads contiguous runs besides its two bodies' pose and solver blocks.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "np_geometry.hpp"
#include "stages.hpp"

namespace nph {

namespace {

// Poses of a manifold's bodies: in HBM (the per-colour kernels) ...
struct GlobalPose {
  DevBodies b;
  __device__ void load(int i, bool, f3& t, q4& q) const {
    t = xyz(b.pos(i));
    q = toq(b.rot(i));
  }
  __device__ void store(int i, f3 t, q4 q) const {
    b.pos(i) = f4(t, 0.0f);
    b.rot(i) = fromq(q);
  }
};

// ... or in LDS for the scene's dynamic bodies, indexed by their rank in the scene (the
// scene-blocked kernel); a static body's pose is read from HBM, and never written.
struct LdsPose {
  DevBodies b;
  float4* pos;
  float4* rot;
  const int* local;
  __device__ void load(int i, bool dyn, f3& t, q4& q) const {
    if (dyn) {
      const int k = local[i];
      t = xyz(pos[k]);
      q = toq(rot[k]);
    } else {
      t = xyz(b.pos(i));
      q = toq(b.rot(i));
    }
  }
  __device__ void store(int i, f3 t, q4 q) const {
    const int k = local[i];
    pos[k] = f4(t, 0.0f);
    rot[k] = fromq(q);
  }
};

// The value of lane `from` of this lane's quad.
__device__ __forceinline__ float quad_get(float v, int from) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute((int(threadIdx.x & 60u) + from) << 2, __float_as_int(v)));
}
__device__ __forceinline__ f3 quad_get(f3 v, int from) {
  return f3{quad_get(v.x, from), quad_get(v.y, from), quad_get(v.z, from)};
}
// The value of the neighbouring lane (0 and 1, 2 and 3 of the quad).
__device__ __forceinline__ float pair_swap(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true));
}

// One manifold on kLanes lanes: on a quad, whose lane k (threadIdx.x & 3) has contact k, or, with one
// contact, on one lane. The four lanes stay together: every branch around an exchange is taken on values they share.
template <int kLanes, bool kMask, class A>
__device__ __forceinline__ void position_lanes(const A& acc, const DevBodies& b, const SimParams& p,
                                               const SolverBufs& sb, int slot) {
  const int k = kLanes == 1 ? 0 : int(threadIdx.x & 3u);
  const int4 q = sb.sinfo[slot];
  const int b1 = q.x & 0x3fffffff, b2 = q.y & 0x3fffffff;
  const bool d1 = (q.x >> 30) & 1;
  const bool d2 = (q.y >> 30) & 1;
  const uint32_t r0 = uint32_t(q.z);
  const int cnt = kLanes == 1 ? 1 : q.w & 7;
  const float4 g1 = sb.pgeo[2 * long(slot)], g2 = sb.pgeo[2 * long(slot) + 1];
  const f3 h1 = xyz(g1), h2 = xyz(g2);
  const float m1 = g1.w, m2 = g2.w;
  const float4* P = sb.prec + 3 * long(r0 + (k < cnt ? k : 0));
  const float4 pa = P[0], pc = P[1], pe = P[2];
  f3 t1, t2;
  q4 q1, q2;
  acc.load(b1, d1, t1, q1);
  acc.load(b2, d2, t2, q2);
  float im1 = 0.0f, im2 = 0.0f;
  m33 I1, I2;
  if (d1) I1 = load_inv(b, b1, im1);
  if (d2) I2 = load_inv(b, b2, im2);
  // jacobian masks (fill_constraint_geometry masks the jacobian, rigid_body.rs:685-705)
  f3 ml1{1.0f, 1.0f, 1.0f}, ma1{1.0f, 1.0f, 1.0f}, ml2{1.0f, 1.0f, 1.0f}, ma2{1.0f, 1.0f, 1.0f};
  if (kMask) {
    b.mask(b1, ml1, ma1);
    b.mask(b2, ml2, ma2);
  }
  const int kind = __float_as_int(pa.w);
  const int k1 = __float_as_int(pc.w), k2 = __float_as_int(pe.w);
  const int quad = threadIdx.x & 60;
  bool moved = false;
  for (int from = 0; from < cnt;) {
    bool act = false;
    f3 l1{0.0f, 0.0f, 0.0f}, a1{0.0f, 0.0f, 0.0f}, l2{0.0f, 0.0f, 0.0f}, a2{0.0f, 0.0f, 0.0f};  // displacements
    if (k >= from && k < cnt) {
      const Contact g = reevaluate(kind, xyz(pa), xyz(pc), xyz(pe), k1, h1, t1, q1, k2, h2, t2, q2);
      const f3 w1 = add(g.w1, scale(g.n, m1));
      const f3 w2 = sub(g.w2, scale(g.n, m2));
      const float depth = (g.depth + m1) + m2;
      const float rhs = fmaxf_((-depth + p.allowed_linear_error) * p.erp, -p.max_linear_correction);
      if (!(rhs >= 0.0f)) {
        float inv_r = 0.0f;
        if (d1) {
          const f3 dir = neg(g.n);
          f3 ang = cross(sub(w1, t1), dir);
          if (kMask) ang = cmul(ang, ma1);
          l1 = scale(kMask ? cmul(dir, ml1) : dir, im1);
          a1 = mulv(I1, ang);
          inv_r = inv_r + (im1 + dot(ang, a1));
        }
        if (d2) {
          const f3 dir = g.n;
          f3 ang = cross(sub(w2, t2), dir);
          if (kMask) ang = cmul(ang, ma2);
          l2 = scale(kMask ? cmul(dir, ml2) : dir, im2);
          a2 = mulv(I2, ang);
          inv_r = inv_r + (im2 + dot(ang, a2));
        }
        if (inv_r != 0.0f) {
          act = true;
          const float r = 1.0f / inv_r;
          const float impulse = -rhs * r;
          l1 = scale(l1, impulse);
          a1 = scale(a1, impulse);
          l2 = scale(l2, impulse);
          a2 = scale(a2, impulse);
        }
      }
    }
    if (kLanes == 1) {
      if (act && d1) apply_displacement(t1, q1, l1, a1);
      if (act && d2) apply_displacement(t2, q2, l2, a2);
      moved = act;
      break;
    }
    const uint32_t acts = uint32_t(__ballot(act) >> quad) & 0xfu;
    if (acts == 0u) break;
    const int f = __ffs(int(acts)) - 1;
    // body 1's pose on the even lanes, body 2's on the odd ones, from the displacements of lane f
    const bool first = (k & 1) == 0;
    const f3 lf1 = quad_get(l1, f), af1 = quad_get(a1, f), lf2 = quad_get(l2, f), af2 = quad_get(a2, f);
    f3 t = pick(first, t1, t2);
    q4 r = pick(first, q1, q2);
    if (first ? d1 : d2) apply_displacement(t, r, pick(first, lf1, lf2), pick(first, af1, af2));
    const f3 to{pair_swap(t.x), pair_swap(t.y), pair_swap(t.z)};
    const q4 ro{pair_swap(r.i), pair_swap(r.j), pair_swap(r.k), pair_swap(r.w)};
    t1 = pick(first, t, to);
    q1 = pick(first, r, ro);
    t2 = pick(first, to, t);
    q2 = pick(first, ro, r);
    moved = true;
    from = f + 1;
  }
  if (moved && k == 0 && d1) acc.store(b1, t1, q1);
  if (moved && k == (kLanes == 1 ? 0 : 1) && d2) acc.store(b2, t2, q2);
}

// The class's manifolds on `lanes` lanes: a quad for each of those with several contacts, a lane for
// each of the others, which start in a wavefront of their own and so run their code alone.
template <bool kMask, class A, class At>
__device__ __forceinline__ void position_class(const A& acc, const DevBodies& b, const SimParams& p,
                                               const SolverBufs& sb, const ClassSpan& c, int lane, int lanes,
                                               const At& at) {
  const int quads = (4 * c.multi + 63) & ~63;
  for (int t = lane; t < quads + c.single; t += lanes) {
    if (t < quads) {
      if (t < 4 * c.multi) position_lanes<4, kMask>(acc, b, p, sb, at(c.first + (t >> 2)));
    } else {
      position_lanes<1, kMask>(acc, b, p, sb, at(c.first + c.multi + t - quads));
    }
  }
}

template <bool kMask>
__global__ void __launch_bounds__(64) k_position(DevBodies b, SimParams p, SolverBufs sb, ClassSpan c) {
  position_class<kMask>(GlobalPose{b}, b, p, sb, c, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x,
                        [](int i) { return i; });
}

// Consecutive small classes of the visiting order in one workgroup, a barrier between classes
// (the same corrections in the same order per body as one launch per class).
template <bool kMask>
__global__ void __launch_bounds__(kRunLanes) k_position_run(DevBodies b, SimParams p, SolverBufs sb, ClassRun run) {
  for (int k = 0; k < run.n; ++k) {
    position_class<kMask>(GlobalPose{b}, b, p, sb, run.r[k], threadIdx.x, blockDim.x, [](int i) { return i; });
    __syncthreads();
  }
}

// Scene-blocked position correction: one workgroup per scene, the scene's dynamic poses in LDS,
// `iterations` passes over the colours in the visiting order with a barrier between colours.
template <int kBlock, int kCap, bool kMask>
__global__ void __launch_bounds__(kBlock) k_position_blocked(DevBodies b, SimParams p, SolverBufs sb, SceneBlocks sc,
                                                           const int* __restrict__ scene_list,
                                                           VisitOrder visit, int iterations) {
  __shared__ float4 s_pos[kCap];
  __shared__ float4 s_rot[kCap];
  const int s = scene_list[blockIdx.x];
  const int d0 = sc.dyn_start[s], nd = sc.dyn_start[s + 1] - d0;
  for (int i = threadIdx.x; i < nd; i += kBlock) {
    const int body = sc.dyn_list[d0 + i];
    s_pos[i] = b.pos(body);
    s_rot[i] = b.rot(body);
  }
  __syncthreads();
  const LdsPose acc{b, s_pos, s_rot, sc.local};
  for (int it = 0; it < iterations; ++it) {
    for (int k = 0; k < visit.n; ++k) {
      position_class<kMask>(acc, b, p, sb, scene_span(sc, visit, s, k), threadIdx.x, kBlock,
                            [&](int i) { return sc.at(i); });
      __syncthreads();
    }
  }
  for (int i = threadIdx.x; i < nd; i += kBlock) {
    const int body = sc.dyn_list[d0 + i];
    b.pos(body) = s_pos[i];
    b.rot(body) = s_rot[i];
  }
}

}  // namespace

void launch_position_colour(const DevBodies& b, const SimParams& p, const ClassSpan& c, SolverBufs& sb,
                            hipStream_t s) {
  // 64-lane workgroups; the grid-stride loop walks what is above the cap
  const long lanes = ((4l * c.multi + 63) & ~63l) + c.single;
  const dim3 grid(unsigned(std::min(std::max((lanes + 63) / 64, 1l), 65536l)));
  if (b.kmask) hipLaunchKernelGGL(k_position<true>, grid, dim3(64), 0, s, b, p, sb, c);
  else hipLaunchKernelGGL(k_position<false>, grid, dim3(64), 0, s, b, p, sb, c);
}

template <bool kMask>
void position_blocked(const DevBodies& b, const SimParams& p, SolverBufs& sb, const SceneBlocks& sc,
                      const VisitOrder& visit, int iterations, int block, hipStream_t s_small, hipStream_t s_large) {
  if (sc.n_large > 0) {
    if (block == 256)
      hipLaunchKernelGGL((k_position_blocked<256, kLdsBodies, kMask>), dim3(sc.n_large), dim3(256), 0, s_large, b, p,
                         sb, sc, sc.large_list, visit, iterations);
    else if (block == 512)
      hipLaunchKernelGGL((k_position_blocked<512, kLdsBodies, kMask>), dim3(sc.n_large), dim3(512), 0, s_large, b, p,
                         sb, sc, sc.large_list, visit, iterations);
    else
      hipLaunchKernelGGL((k_position_blocked<1024, kLdsBodies, kMask>), dim3(sc.n_large), dim3(1024), 0, s_large, b,
                         p, sb, sc, sc.large_list, visit, iterations);
  }
  if (sc.n_small > 0)
    hipLaunchKernelGGL((k_position_blocked<kSmallLanes, kSmallScene, kMask>), dim3(sc.n_small), dim3(kSmallLanes), 0,
                       s_small, b, p, sb, sc, sc.small_list, visit, iterations);
}

void launch_position_blocked(const DevBodies& b, const SimParams& p, SolverBufs& sb, const SceneBlocks& sc,
                             const VisitOrder& visit, int iterations, int block, hipStream_t s_small,
                             hipStream_t s_large) {
  if (b.kmask) position_blocked<true>(b, p, sb, sc, visit, iterations, block, s_small, s_large);
  else position_blocked<false>(b, p, sb, sc, visit, iterations, block, s_small, s_large);
}

void launch_position_run(const DevBodies& b, const SimParams& p, SolverBufs& sb, const ClassRun& run, hipStream_t s) {
  // as many lanes as the largest class takes: fewer waves meet at each barrier
  int lanes = 64;
  for (int k = 0; k < run.n; ++k) lanes = std::max(lanes, ((4 * run.r[k].multi + 63) & ~63) + run.r[k].single);
  const dim3 block(unsigned(std::min((lanes + 63) & ~63, kRunLanes)));
  if (b.kmask) hipLaunchKernelGGL(k_position_run<true>, dim3(1), block, 0, s, b, p, sb, run);
  else hipLaunchKernelGGL(k_position_run<false>, dim3(1), block, 0, s, b, p, sb, run);
}

}  // namespace nph
