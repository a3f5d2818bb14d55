// nphysics_amd/csrc/world.hip -- host orchestration of one MechanicalWorld::step on one GPU and
// the C ABI of include/nphys.h.
//
// Step order (src/world/mechanical_world.rs:199-396):
//   1. collision detection on the current poses when bodies were added or moved by the caller
//      (:250-253);
//   2. per-body dynamics, accelerations, ext = dt acc, dv = 0 (k_prestep; :230-243 and
//      moreau_jean_solver.rs:137-174);
//   3. MoreauJeanSolver::step (moreau_jean_solver.rs:47-90): colouring, assembly with warm start,
//      coloured SOR-Prox sweeps, residual, impulse cache, integration, coloured position
//      correction;
//   4. the CCD-phase sync + broad phase over swept AABBs (:604-606), the final sync (a no-op for
//      the loose AABBs, checked anyway) and the broad + narrow phase that produce the next step's
//      manifolds (:375-385).
// The host reads back a handful of counters per step (loose-AABB changes, pair/contact totals,
// colouring progress, colour offsets, residual partials); everything else stays on the device.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <initializer_list>
#include <limits>
#include <map>
#include <cstdlib>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "../../include/nphys.h"
#include "common.hpp"
#include "devmath.hpp"
#include "kernels.hpp"
#include "mlp.hpp"
#include "stages.hpp"

namespace nph {

namespace {

// Manifold list plus the contact slots of every broad-phase pair (kPairSlots per pair).
struct ContactBufs {
  DBuf mbody, mfirst, mcount, rec, imp, bfirst;
  int M = 0, C = 0, nb = 0;  // nb: bodies covered by bfirst
  hipError_t ensure(size_t mcap, size_t slots) {
    hipError_t e;
    if ((e = mbody.ensure(mcap * sizeof(int2))) != hipSuccess) return e;
    if ((e = mfirst.ensure(mcap * 4)) != hipSuccess) return e;
    if ((e = mcount.ensure(mcap * 4)) != hipSuccess) return e;
    if ((e = rec.ensure(slots * kContactFields * sizeof(float4))) != hipSuccess) return e;
    if ((e = imp.ensure(slots * sizeof(float4))) != hipSuccess) return e;
    return hipSuccess;
  }
  DevContacts view() const {
    DevContacts d;
    d.mbody = mbody.as<int2>();
    d.mfirst = mfirst.as<int>();
    d.mcount = mcount.as<int>();
    d.rec = rec.as<float4>();
    d.imp = imp.as<float4>();
    d.bfirst = nb > 0 ? bfirst.as<int>() : nullptr;
    d.bcount = nb;
    return d;
  }
};

enum StageEv { EV_START, EV_PRE_CD, EV_ASM, EV_VEL, EV_INT, EV_POS, EV_CCD, EV_BP, EV_NP, EV_COUNT };

// Small device values to pinned host memory without a stream synchronisation: one workgroup copies
// up to four word ranges into the host buffer, fences at system scope and then writes the
// sequence number the host waits for. Launched last in stream order, so the flag also means that
// everything enqueued before it has completed.
struct RbJob {
  const uint32_t* src[4];
  int n[4];
  int dst[4];
};

__global__ void __launch_bounds__(256) k_readback(RbJob j, uint32_t* host, int flag, uint32_t seq) {
  for (int s = 0; s < 4; ++s)
    for (int i = threadIdx.x; i < j.n[s]; i += blockDim.x) host[j.dst[s] + i] = j.src[s][i];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(host + flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

struct World {
  hipStream_t stream = nullptr;
  // the scene-blocked solve runs its large scenes on stream_large beside the small ones on stream
  // (fork and join by events)
  hipStream_t stream_large = nullptr;
  hipEvent_t fork_ev = nullptr, join_ev = nullptr;
  int device = 0;
  nphys_params prm{};
  SimParams sp{};
  int32_t contact_model = NPHYS_CONTACT_MODEL_SIGNORINI_COULOMB_PYRAMID;

  // host copies of the per-body static attributes
  std::vector<int> h_status, h_shape, h_scene;
  int scene_bits = 0;  // bits of the scene index above the Morton code (0: one scene)
  std::vector<float4> h_dims, h_local_i;
  std::vector<float> h_margin, h_qlim, h_friction, h_restitution, h_mass;
  int n = 0;

  // device body arrays
  DBuf status, shape, scene, dims, margin, qlim, friction, restitution, mass, local_i;
  DBuf pose;  // kPoseBlock float4 per body: position, rotation
  DBuf sol;   // kSolverBlock float4 per body: inverse inertia and mass, solver velocity increment
  DBuf pos0, rot0, linvel, angvel, ext_lin, ext_ang;
  DBuf loose_mn, loose_mx;
  DBuf act;  // float2 per body: activation energy (0: asleep), sleep threshold (< 0: never sleeps)
  // Optional per-body attributes (damping and clamps, flags, material ids, surface velocities);
  // each is passed to the kernels only when some body differs from the default.
  std::vector<float4> h_damp, h_surf;
  std::vector<uint4> h_groups;
  std::vector<int> h_flags, h_matid;
  bool any_damp = false, any_flags = false, any_mask = false, any_matid = false, any_surf = false;
  bool any_groups = false;
  DBuf damp, bflags, matid, surf, groups;
  // External forces accumulated for the next step (cleared after it), the angular velocity of the
  // last dynamics update, and the rotations from before a set_state of the current interval.
  DBuf f_lin, f_ang, w_dyn, rot_dyn, af_tmp;
  bool forces_pending = false, rot_dyn_saved = false;
  // material coefficient table (sorted keys min id << 32 | max id), friction and restitution
  std::vector<std::pair<unsigned long long, float>> mt_host[2];
  DBuf mt_key[2], mt_val[2];
  // Sleeping: on once a dynamic body with a threshold exists; a wake of every sleeping body is
  // due at the next step after the caller set the bodies' state.
  bool sleeping = false, wake_pending = false;
  int64_t n_dynamic = 0, active_bodies = 0;
  DBuf act_parent, act_can, act_touch, act_pos, act_mflag[2], sl_mbody[2], sl_mfirst[2], sl_mcount[2];

  ScanState scan;  // prefix sums on `stream`

  // broad phase
  DBuf bp_dirty, bp_list;
  // The segments of the last search stand; searches by the present order (sorted anew every
  // kOrderAge-th, and when the bodies were added or moved by the caller).
  bool segments_valid = false;
  bool incremental_bp = true;
  static constexpr int kOrderAge = 16;
  int order_age = kOrderAge;
  // Detections in a row, without and with a narrow phase, that replaced no loose AABB (up to kCalm), and the pair
  // capacity of the narrow phase's lists of the present pairs (0: there are none).
  static constexpr int kCalm = 2;
  int calm[2] = {0, 0};
  int list_room = 0;
  DBuf bp_small, keys, vals, keys_alt, vals_alt, leaf_mn, leaf_mx, box_mn, box_mx, box_top, cand, cand_count, pairs,
      bp_tmp;
  int cap = 32;
  int npairs = 0;
  bool pairs_dirty = true;
  // Pairs a narrow phase takes: a manifold's first slot is packed in 28 bits of the solver's slot record.
  static constexpr int kMostPairs = (1 << 28) / kPairSlots - 1;
  int most_pairs = kMostPairs;
  bool moved = true;
  // the next step starts with collision detection: collision groups changed, or the last detection failed
  bool recollide = false;

  // narrow phase
  DBuf np_count, np_perm;
  DBuf rd_moff, rd_rec, rd_imp;  // contact readback staging
  ContactBufs cb[2];
  int cur = 0;      // index of the manifolds produced by the last collision detection
  bool have_solved = false;

  // solver
  // The manifolds handed to the solver with cb[k]'s contacts: all of cb[k], or (sleeping) the
  // compacted list of those with an awake dynamic side in sl_*[k].
  DevContacts sview[2] = {};
  int sview_M[2] = {0, 0}, sview_C[2] = {0, 0};
  bool sview_compact[2] = {false, false};
  DBuf sv_state2[2];  // colouring state of the manifolds of sview[k]
  DBuf sv_deg, sv_adj_off, sv_adj, sv_place, sv_hist, sv_ckeys, sv_col_start, sv_slot_of, sv_sinfo, sv_rec, sv_lam,
      sv_has, sv_prec, sv_pgeo, sv_tmp;
  int ncolours = 0;
  long rec_stride = 0;
  int colour_rounds = 0;
  // colouring rounds enqueued before the host looks: what the last solve took (a step's, a CCD substep's) and one
  // more, within these bounds
  static constexpr int kMinRounds = 4, kMaxRounds = 32;
  int round_batch[2] = {kMinRounds, kMinRounds};
  // solves left for which a world too crowded for k_colour_small goes by it
  static constexpr int kCrowdedSolves = 16;
  int crowded[2] = {0, 0};
  std::vector<int> colour_visit;  // colour classes in visiting order
  long solve_count = 0;    // solves performed, never reset
  std::vector<ClassSpan> h_span;    // their slots, in that order
  bool split_order = false;        // classes list manifolds with several contacts first
  std::vector<int> class_contacts;  // and their contacts
  int solved_M = 0, solved_C = 0;
  double res_inf = 0.0, res_rms = 0.0;
  double *red_host = nullptr, *red_dev = nullptr;  // residual partials (pinned, device-mapped)
  size_t red_cap = 0;
  int res_pending_blocks = -1, res_pending_C = 0;
  // solve-to-residual mode (off when res_target <= 0): see nphys_set_residual_target
  double res_target = 0.0;
  int res_max_sweeps = 500, res_check_every = 1, res_norm = NPHYS_RESIDUAL_MAX;
  int last_sweeps = 0;
  // learned warm start: network (FP32 parameters + BF16 images), per-record features, impulse
  // units, predictions and recorded targets; the judge's saved plain solve
  // scene-blocked solve: per-scene dynamic-body lists (host-built at insertion), the per-solve
  // scene-major slot order, and the variant chosen by the autotuner (0 per-colour launches,
  // 256/512/1024 the blocked kernels' workgroup size for the scenes of more than 256 dynamic bodies)
  int nscenes = 1, max_scene_dyn = 0;
  // end of the last non-dynamic body, and which kinds of pairs can occur (a cuboid-cuboid pair has a
  // dynamic cuboid)
  int fixed_end = 0;
  bool any_cuboid = false, any_ball = false;
  DBuf sc_dyn_start, sc_dyn_list, sc_local, sc_keys, sc_slot, sc_keys_alt, sc_slot_alt, sc_start, sc_info, sc_rank, sc_small,
      sc_large;
  int n_small_scenes = 0, n_large_scenes = 0;
  int variant_request = -1;  // -1: autotune; else forced
  int cur_variant = 0;
  static constexpr int kTuneReps = 3;
  std::vector<int> tune_cands;
  std::vector<double> tune_time;
  std::vector<int> tune_count;
  bool tuned = false, tune_pending = false;
  int tune_M = 0;  // manifold count when the current pick was timed
  hipEvent_t tune_ev[2] = {nullptr, nullptr};
  bool ml_loaded = false, capture = false, judge = false;
  long samples = 0;
  DBuf ml_params, ml_img, ml_X, ml_ls, ml_y, ml_t, jd_lam, jd_lam0, jd_dv;
  std::vector<int> last_colours;
  bool keep_colours = false;

  // joints: static per-joint arrays (host copies in joint order), their greedy colouring with the
  // joints listed colour by colour, per-solve row records and impulses, and the judge's saved ones
  std::vector<int4> h_jinfo;
  std::vector<float4> h_ja1, h_ja2, h_jf1, h_jf2;
  std::vector<float2> h_jbrk;
  std::vector<int> h_jorder;
  std::vector<int2> h_jcrange;
  int nj = 0, njcol = 0;
  DBuf j_info, j_a1, j_a2, j_f1, j_f2, j_brk, j_imp_lin, j_imp_ang, j_state, j_order, j_crange, j_rec, j_lam, jd_jlam;

  // CCD, once some body is CCD-enabled: per-body flags (bit 0 ccd_enabled, bit 1 linear motion
  // interpolation) and keys (a static collider that shares a static body takes the index of that
  // body's first collider), the CcdBufs arrays, the scratch manifolds of the island rounds, and the
  // last prediction's results
  bool any_ccd = false;
  std::vector<int> h_ccd, h_ccd_key;
  std::map<std::pair<int, int>, int> static_owner;  // (scene, static body index) -> first collider
  DBuf ccd_flags, ccd_keys, ccd_rot, ccd_time, ccd_frozen, ccd_slot, ccd_queue, ccd_seen, ccd_seen_at, ccd_group, ccd_stage, ccd_imp, ccd_ctl,
      ccd_in, ccd_new, ccd_prep, ccd_prepared, ccd_eval, ccd_kept, ccd_cand, ccd_cpos, ccd_list, ccd_lpair,
      ccd_deg, ccd_off, ccd_fill, ccd_adj, ccd_bodies, ccd_sbodies;
  ContactBufs ccd_cb;
  int ccd_cap = 0, ccd_nimp = 0;
  float ccd_last_toi = 0.0f, ccd_min_over = 0.0f;
  bool ccd_sub = false;        // a CCD substep is being solved: no joint rows, per-colour launches
  float dyn_dt_next = 0.0f;    // time step of the bodies' last dynamics update (a substep's after one)

  // Readback buffer (pinned, device-mapped, coherent): words [0, 64) small per-step values,
  // [kRbClass, +2 (kMaxColours + 2)) the class offsets, kRbFlag the sequence flag.
  static constexpr int kRbClass = 64, kRbFlag = kRbClass + 2 * (kMaxColours + 2) + 64, kRbWords = kRbFlag + 64;
  uint32_t* rb_host = nullptr;
  uint32_t* rb_dev = nullptr;
  uint32_t rb_seq = 0;
  // Staging of set_state and get_state (pinned, device-mapped): 52 B per body, grown on first use.
  float *io_host = nullptr, *io_dev = nullptr;
  size_t io_cap = 0;
  struct RbSeg {
    const uint32_t* src;
    int n;
    int dst;
  };
  hipEvent_t ev[EV_COUNT] = {};
  nphys_counters counters{};
  bool counters_enabled = false;
  std::vector<hipEvent_t> kt_ev;  // event pairs around sweep-kernel launches
  int kt_used = 0;

  ~World() {
    if (red_host) (void)hipHostFree(red_host);
    if (rb_host) (void)hipHostFree(rb_host);
    if (io_host) (void)hipHostFree(io_host);
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
    for (auto& e : kt_ev)
      if (e) (void)hipEventDestroy(e);
    for (auto& e : tune_ev)
      if (e) (void)hipEventDestroy(e);
    for (auto& e : ml_ev)
      if (e) (void)hipEventDestroy(e);
    if (fork_ev) (void)hipEventDestroy(fork_ev);
    if (join_ev) (void)hipEventDestroy(join_ev);
    if (stream_large) (void)hipStreamDestroy(stream_large);
    if (stream) (void)hipStreamDestroy(stream);
  }

  void set_params(const nphys_params& p) {
    prm = p;
    sp.dt = float(p.dt);
    sp.inv_dt = sp.dt == 0.0f ? 0.0f : 1.0f / sp.dt;
    sp.erp = float(p.erp);
    sp.warmstart_coeff = float(p.warmstart_coeff);
    sp.restitution_threshold = float(p.restitution_velocity_threshold);
    sp.allowed_linear_error = float(p.allowed_linear_error);
    sp.max_linear_correction = float(p.max_linear_correction);
    sp.allowed_angular_error = float(p.allowed_angular_error);
    sp.max_angular_correction = float(p.max_angular_correction);
    sp.gx = float(p.gravity[0]);
    sp.gy = float(p.gravity[1]);
    sp.gz = float(p.gravity[2]);
    sp.dyn_dt = sp.dt;
    dyn_dt_next = sp.dt;
  }

  int init(const nphys_params& p) {
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
      return set_err(NPHYS_ERR_NO_DEVICE, "no HIP device");
    HIPCK(hipGetDevice(&device));
    HIPCK(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    HIPCK(hipStreamCreateWithFlags(&stream_large, hipStreamNonBlocking));
    HIPCK(hipEventCreateWithFlags(&fork_ev, hipEventDisableTiming));
    HIPCK(hipEventCreateWithFlags(&join_ev, hipEventDisableTiming));
    HIPCK(hipHostMalloc(reinterpret_cast<void**>(&rb_host), kRbWords * sizeof(uint32_t),
                        hipHostMallocMapped | hipHostMallocCoherent));
    std::memset(rb_host, 0, kRbWords * sizeof(uint32_t));
    HIPCK(hipHostGetDevicePointer(reinterpret_cast<void**>(&rb_dev), rb_host, 0));
    for (auto& e : ev) HIPCK(hipEventCreate(&e));
    for (auto& e : tune_ev) HIPCK(hipEventCreate(&e));
    set_params(p);
    HIPCK(bp_small.ensure(64 * sizeof(uint32_t)));
    return NPHYS_OK;
  }

  DevBodies bodies() const {
    DevBodies b;
    b.n = n;
    b.status = status.as<int>();
    b.shape = shape.as<int>();
    b.scene = scene.as<int>();
    b.dims = dims.as<float4>();
    b.margin = margin.as<float>();
    b.qlim = qlim.as<float>();
    b.friction = friction.as<float>();
    b.restitution = restitution.as<float>();
    b.mass = mass.as<float>();
    b.local_i = local_i.as<float4>();
    b.pose = pose.as<float4>();
    b.sol = sol.as<float4>();
    b.pos0 = pos0.as<float4>();
    b.rot0 = rot0.as<float4>();
    b.linvel = linvel.as<float4>();
    b.angvel = angvel.as<float4>();
    b.ext_lin = ext_lin.as<float4>();
    b.ext_ang = ext_ang.as<float4>();
    b.loose_mn = loose_mn.as<float4>();
    b.loose_mx = loose_mx.as<float4>();
    b.act = sleeping ? act.as<float2>() : nullptr;
    b.damp = any_damp ? damp.as<float4>() : nullptr;
    b.flags = any_flags ? bflags.as<int>() : nullptr;
    b.kmask = any_mask ? bflags.as<int>() : nullptr;
    b.mat_id = any_matid ? matid.as<int>() : nullptr;
    b.surf_vel = any_surf ? surf.as<float4>() : nullptr;
    b.f_lin = forces_pending ? f_lin.as<float4>() : nullptr;
    b.f_ang = forces_pending ? f_ang.as<float4>() : nullptr;
    b.w_dyn = w_dyn.as<float4>();
    b.ccd = any_ccd ? ccd_flags.as<int>() : nullptr;
    b.ccd_key = any_ccd ? ccd_keys.as<int>() : nullptr;
    b.ccd_rot = any_ccd ? ccd_rot.as<float4>() : nullptr;
    b.groups = any_groups ? groups.as<uint4>() : nullptr;
    return b;
  }

  MatTable mat_table() const {
    MatTable t;
    t.fkey = mt_key[0].as<unsigned long long>();
    t.fval = mt_val[0].as<float>();
    t.nf = int(mt_host[0].size());
    t.rkey = mt_key[1].as<unsigned long long>();
    t.rval = mt_val[1].as<float>();
    t.nr = int(mt_host[1].size());
    return t;
  }

  // ------------------------------------------------------------------ scene
  JointBufs joint_view() {
    JointBufs j;
    j.nj = nj;
    j.ncol = njcol;
    j.info = j_info.as<int4>();
    j.a1 = j_a1.as<float4>();
    j.a2 = j_a2.as<float4>();
    j.f1 = j_f1.as<float4>();
    j.f2 = j_f2.as<float4>();
    j.brk = j_brk.as<float2>();
    j.imp_lin = j_imp_lin.as<float4>();
    j.imp_ang = j_imp_ang.as<float4>();
    j.state = j_state.as<int>();
    j.order = j_order.as<int>();
    j.crange = j_crange.as<int2>();
    j.rec = j_rec.as<float4>();
    j.lam = j_lam.as<float4>();
    return j;
  }

  // Greedy colouring of the joints in joint order: a joint takes the smallest colour that no
  // earlier joint sharing one of its dynamic bodies has (the CPU restatement colours the same way).
  void colour_joints() {
    std::vector<std::vector<int>> used(size_t(std::max(n, 1)));
    njcol = 0;
    for (int ji = 0; ji < nj; ++ji) {
      int4& inf = h_jinfo[size_t(ji)];
      std::vector<char> taken;
      for (int bi : {inf.y, inf.z}) {
        if (h_status[size_t(bi)] != NPHYS_STATUS_DYNAMIC) continue;
        for (int c : used[size_t(bi)]) {
          if (int(taken.size()) <= c) taken.resize(size_t(c) + 1, 0);
          taken[size_t(c)] = 1;
        }
      }
      int c = 0;
      while (c < int(taken.size()) && taken[size_t(c)]) ++c;
      inf.w = c;
      njcol = std::max(njcol, c + 1);
      for (int bi : {inf.y, inf.z})
        if (h_status[size_t(bi)] == NPHYS_STATUS_DYNAMIC) used[size_t(bi)].push_back(c);
    }
    h_jorder.clear();
    h_jcrange.assign(size_t(njcol), int2{0, 0});
    for (int c = 0; c < njcol; ++c) {
      h_jcrange[size_t(c)].x = int(h_jorder.size());
      for (int ji = 0; ji < nj; ++ji)
        if (h_jinfo[size_t(ji)].w == c) h_jorder.push_back(ji);
      h_jcrange[size_t(c)].y = int(h_jorder.size()) - h_jcrange[size_t(c)].x;
    }
  }

  // JointConstraintSet::insert for every joint of the descriptor (ball_constraint.rs:27-48,
  // fixed_constraint.rs:28-58, revolute_constraint.rs:37-72).
  int add_joints(const nphys_joint_desc& d, int32_t* first) {
    if (d.n < 0 || (d.n > 0 && (!d.kind || !d.body1 || !d.body2 || !d.anchor1 || !d.anchor2)))
      return set_err(NPHYS_ERR_INVALID, "bad joint descriptor");
    for (int i = 0; i < d.n; ++i) {
      const int b1 = d.body1[i], b2 = d.body2[i];
      if (b1 < 0 || b1 >= n || b2 < 0 || b2 >= n || b1 == b2) return set_err(NPHYS_ERR_INVALID, "bad joint body");
      if (d.kind[i] < NPHYS_JOINT_BALL || d.kind[i] > NPHYS_JOINT_CYLINDRICAL)
        return set_err(NPHYS_ERR_INVALID, "bad joint kind");
      if (h_status[size_t(b1)] != NPHYS_STATUS_DYNAMIC && h_status[size_t(b2)] != NPHYS_STATUS_DYNAMIC)
        return set_err(NPHYS_ERR_INVALID, "a joint needs a dynamic body");
    }
    if (first) *first = nj;
    if (d.n == 0) return NPHYS_OK;
    HIPCK(hipStreamSynchronize(stream));
    const int old = nj;
    for (int i = 0; i < d.n; ++i) {
      h_jinfo.push_back(make_int4(d.kind[i], d.body1[i], d.body2[i], 0));
      h_ja1.push_back(make_float4(d.anchor1[3 * i], d.anchor1[3 * i + 1], d.anchor1[3 * i + 2], 0.0f));
      h_ja2.push_back(make_float4(d.anchor2[3 * i], d.anchor2[3 * i + 1], d.anchor2[3 * i + 2], 0.0f));
      float4 f1 = make_float4(0.0f, 0.0f, 0.0f, 1.0f), f2 = f1;
      if (d.kind[i] == NPHYS_JOINT_FIXED) {
        if (d.frame1) f1 = make_float4(d.frame1[4 * i], d.frame1[4 * i + 1], d.frame1[4 * i + 2], d.frame1[4 * i + 3]);
        if (d.frame2) f2 = make_float4(d.frame2[4 * i], d.frame2[4 * i + 1], d.frame2[4 * i + 2], d.frame2[4 * i + 3]);
      } else if (d.kind[i] == NPHYS_JOINT_PRISMATIC) {
        f1 = d.axis1 ? make_float4(d.axis1[3 * i], d.axis1[3 * i + 1], d.axis1[3 * i + 2], 0.0f)
                     : make_float4(0.0f, 0.0f, 1.0f, 0.0f);
      } else if (d.kind[i] == NPHYS_JOINT_REVOLUTE || d.kind[i] == NPHYS_JOINT_CYLINDRICAL) {
        f1 = d.axis1 ? make_float4(d.axis1[3 * i], d.axis1[3 * i + 1], d.axis1[3 * i + 2], 0.0f)
                     : make_float4(0.0f, 0.0f, 1.0f, 0.0f);
        f2 = d.axis2 ? make_float4(d.axis2[3 * i], d.axis2[3 * i + 1], d.axis2[3 * i + 2], 0.0f)
                     : make_float4(0.0f, 0.0f, 1.0f, 0.0f);
      }
      h_jf1.push_back(f1);
      h_jf2.push_back(f2);
      const float bf = d.break_force ? d.break_force[i] : -1.0f;
      const float bt = d.break_torque ? d.break_torque[i] : -1.0f;
      h_jbrk.push_back(make_float2(bf >= 0.0f ? bf * bf : FLT_MAX, bt >= 0.0f ? bt * bt : FLT_MAX));
    }
    nj += d.n;
    colour_joints();
    const size_t J = size_t(nj);
    HIPCK(j_info.ensure(J * sizeof(int4)));
    HIPCK(j_a1.ensure(J * sizeof(float4)));
    HIPCK(j_a2.ensure(J * sizeof(float4)));
    HIPCK(j_f1.ensure(J * sizeof(float4)));
    HIPCK(j_f2.ensure(J * sizeof(float4)));
    HIPCK(j_brk.ensure(J * sizeof(float2)));
    HIPCK(j_order.ensure(J * sizeof(int)));
    HIPCK(j_crange.ensure(size_t(std::max(njcol, 1)) * sizeof(int2)));
    HIPCK(j_rec.ensure(J * kJointRec * sizeof(float4)));
    HIPCK(j_lam.ensure(J * 2 * sizeof(float4)));
    // cached impulses and broken / removed flags live on the device: kept, the new ones cleared
    HIPCK(j_imp_lin.ensure(J * sizeof(float4), true, stream));
    HIPCK(j_imp_ang.ensure(J * sizeof(float4), true, stream));
    HIPCK(j_state.ensure(J * sizeof(int), true, stream));
    const size_t add = size_t(d.n);
    HIPCK(hipMemsetAsync(j_imp_lin.as<float4>() + old, 0, add * sizeof(float4), stream));
    HIPCK(hipMemsetAsync(j_imp_ang.as<float4>() + old, 0, add * sizeof(float4), stream));
    HIPCK(hipMemsetAsync(j_state.as<int>() + old, 0, add * sizeof(int), stream));
    HIPCK(hipMemcpyAsync(j_info.p, h_jinfo.data(), J * sizeof(int4), hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(j_a1.p, h_ja1.data(), J * sizeof(float4), hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(j_a2.p, h_ja2.data(), J * sizeof(float4), hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(j_f1.p, h_jf1.data(), J * sizeof(float4), hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(j_f2.p, h_jf2.data(), J * sizeof(float4), hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(j_brk.p, h_jbrk.data(), J * sizeof(float2), hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(j_order.p, h_jorder.data(), J * sizeof(int), hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(j_crange.p, h_jcrange.data(), size_t(njcol) * sizeof(int2), hipMemcpyHostToDevice, stream));
    HIPCK(hipStreamSynchronize(stream));
    return NPHYS_OK;
  }

  // JointConstraintSet::remove: the joint no longer takes part in the solve or the islands.
  int remove_joint(int ji) {
    if (ji < 0 || ji >= nj) return set_err(NPHYS_ERR_INVALID, "bad joint handle");
    int st = 0;
    HIPCK(hipMemcpyAsync(&st, j_state.as<int>() + ji, sizeof(int), hipMemcpyDeviceToHost, stream));
    HIPCK(hipStreamSynchronize(stream));
    st |= 2;
    HIPCK(hipMemcpyAsync(j_state.as<int>() + ji, &st, sizeof(int), hipMemcpyHostToDevice, stream));
    HIPCK(hipStreamSynchronize(stream));
    return NPHYS_OK;
  }

  int read_joints(float* lin, float* ang, int32_t* broken, int64_t cap) {
    if (cap < nj) return set_err(NPHYS_ERR_CAPACITY, "joint buffers too small");
    if (nj == 0) return NPHYS_OK;
    const size_t J = static_cast<size_t>(nj);
    std::vector<float4> l(J), a(J);
    std::vector<int> st(J);
    HIPCK(hipMemcpyAsync(l.data(), j_imp_lin.p, J * sizeof(float4), hipMemcpyDeviceToHost, stream));
    HIPCK(hipMemcpyAsync(a.data(), j_imp_ang.p, J * sizeof(float4), hipMemcpyDeviceToHost, stream));
    HIPCK(hipMemcpyAsync(st.data(), j_state.p, J * sizeof(int), hipMemcpyDeviceToHost, stream));
    HIPCK(hipStreamSynchronize(stream));
    for (int i = 0; i < nj; ++i) {
      if (lin) {
        lin[3 * i] = l[size_t(i)].x;
        lin[3 * i + 1] = l[size_t(i)].y;
        lin[3 * i + 2] = l[size_t(i)].z;
      }
      if (ang) {
        ang[3 * i] = a[size_t(i)].x;
        ang[3 * i + 1] = a[size_t(i)].y;
        ang[3 * i + 2] = a[size_t(i)].z;
      }
      if (broken) broken[i] = st[size_t(i)] & 1;
    }
    return NPHYS_OK;
  }

  int add_bodies(const nphys_body_desc& d, int32_t* first) {
    if (d.n < 0) return set_err(NPHYS_ERR_INVALID, "negative body count");
    if (!d.status || !d.shape || !d.dims || !d.pos || !d.rot || !d.density || !d.margin ||
        !d.linear_prediction || !d.friction || !d.restitution)
      return set_err(NPHYS_ERR_INVALID, "missing body array");
    if (int64_t(n) + d.n >= (int64_t(1) << 24)) return set_err(NPHYS_ERR_INVALID, "too many bodies");
    if (first) *first = n;
    if (d.n == 0) return NPHYS_OK;
    const int n0 = n, n1 = n + d.n;
    std::vector<float4> hp(size_t(d.n) * kPoseBlock), hv(d.n), hw(d.n), hmn(d.n), hmx(d.n);
    std::vector<float2> ha(d.n);
    bool any_sleeper = false;
    int64_t new_dynamic = 0;
    for (int k = 0; k < d.n; ++k) {
      const int st = d.status[k], sh = d.shape[k];
      if (st != NPHYS_STATUS_DYNAMIC && st != NPHYS_STATUS_STATIC)
        return set_err(NPHYS_ERR_INVALID, "bad body status");
      if (sh != NPHYS_SHAPE_BALL && sh != NPHYS_SHAPE_CUBOID) return set_err(NPHYS_ERR_INVALID, "bad shape");
      if (d.scene && (d.scene[k] < 0 || d.scene[k] >= NPHYS_MAX_SCENES))
        return set_err(NPHYS_ERR_INVALID, "scene index out of range");
      const float* dm = d.dims + 3 * k;
      if (sh == NPHYS_SHAPE_BALL ? !(dm[0] > 0.0f) : !(dm[0] > 0.0f && dm[1] > 0.0f && dm[2] > 0.0f))
        return set_err(NPHYS_ERR_INVALID, "shape dimensions must be positive");
      if ((d.friction_combine && (d.friction_combine[k] < 0 || d.friction_combine[k] > 3)) ||
          (d.restitution_combine && (d.restitution_combine[k] < 0 || d.restitution_combine[k] > 3)))
        return set_err(NPHYS_ERR_INVALID, "bad combine mode");
    }
    for (int k = 0; k < d.n; ++k) {
      const int st = d.status[k], sh = d.shape[k];
      const float* dm = d.dims + 3 * k;
      const float4 he = sh == NPHYS_SHAPE_BALL ? make_float4(dm[0], dm[0], dm[0], 0.0f)
                                               : make_float4(dm[0], dm[1], dm[2], 0.0f);
      // mass properties (volumetric_ball.rs:9-44, volumetric_cuboid.rs:10-75, volumetric.rs:46-59)
      float m = 0.0f;
      float4 li = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      const float density = d.density[k];
      if (st == NPHYS_STATUS_DYNAMIC && density != 0.0f) {
        if (sh == NPHYS_SHAPE_BALL) {
          const float r = dm[0];
          const float vol = ((((float)M_PI * r) * r) * r) * (float)(4.0 / 3.0);
          m = vol * density;
          const float diag = (r * r) * (float)(2.0 / 5.0);
          li = make_float4(diag * m, diag * m, diag * m, 0.0f);
        } else {
          float vol = 1.0f;
          vol = vol * dm[0] * 2.0f;
          vol = vol * dm[1] * 2.0f;
          vol = vol * dm[2] * 2.0f;
          m = vol * density;
          const float w = ((float)(1.0 / 12.0) * 2.0f) * 2.0f;
          const float ix = (w * dm[0]) * dm[0], iy = (w * dm[1]) * dm[1], iz = (w * dm[2]) * dm[2];
          li = make_float4((iy + iz) * m, (ix + iz) * m, (ix + iy) * m, 0.0f);
        }
      }
      h_status.push_back(st);
      h_shape.push_back(sh);
      h_scene.push_back(d.scene ? d.scene[k] : 0);
      h_dims.push_back(he);
      h_local_i.push_back(li);
      h_mass.push_back(m);
      h_margin.push_back(d.margin[k]);
      h_qlim.push_back(d.margin[k] + d.linear_prediction[k]);
      h_friction.push_back(d.friction[k]);
      h_restitution.push_back(d.restitution[k]);
      // RigidBodyDesc / BasicMaterial attributes (rigid_body.rs:972-990, basic_material.rs:33-43)
      const float fmax = 3.402823466e38f;
      const float4 dp = make_float4(d.linear_damping ? d.linear_damping[k] : 0.0f,
                                    d.angular_damping ? d.angular_damping[k] : 0.0f,
                                    d.max_linear_velocity ? d.max_linear_velocity[k] : fmax,
                                    d.max_angular_velocity ? d.max_angular_velocity[k] : fmax);
      h_damp.push_back(dp);
      any_damp = any_damp || dp.x != 0.0f || dp.y != 0.0f || dp.z != fmax || dp.w != fmax;
      const int kin = d.kinematic_dofs ? (d.kinematic_dofs[k] & 63) : 0;
      const int fl = kin | ((d.gravity_enabled && !d.gravity_enabled[k]) ? kFlagNoGravity : 0) |
                     ((d.friction_combine ? d.friction_combine[k] : 0) << 8) |
                     ((d.restitution_combine ? d.restitution_combine[k] : 0) << 10);
      h_flags.push_back(fl);
      any_flags = any_flags || fl != 0;
      any_mask = any_mask || (st == NPHYS_STATUS_DYNAMIC && kin != 0);
      const int mid = d.material_id ? (d.material_id[k] < 0 ? -1 : d.material_id[k]) : -1;
      h_matid.push_back(mid);
      any_matid = any_matid || mid >= 0;
      const float4 sv = d.surface_velocity
                            ? make_float4(d.surface_velocity[3 * k], d.surface_velocity[3 * k + 1],
                                          d.surface_velocity[3 * k + 2], 0.0f)
                            : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      h_surf.push_back(sv);
      any_surf = any_surf || sv.x != 0.0f || sv.y != 0.0f || sv.z != 0.0f;
      // ColliderDesc::collision_groups: groups 0-29 (CollisionGroups::new() without the array)
      constexpr uint32_t kAllGroups = (1u << 30) - 1u;
      const uint4 cg = d.collision_groups
                           ? make_uint4(d.collision_groups[3 * k] & kAllGroups, d.collision_groups[3 * k + 1] & kAllGroups,
                                        d.collision_groups[3 * k + 2] & kAllGroups, 0u)
                           : make_uint4(kAllGroups, kAllGroups, 0u, 0u);
      h_groups.push_back(cg);
      any_groups = any_groups || cg.x != kAllGroups || cg.y != kAllGroups || cg.z != 0u;
      // ColliderDesc::ccd_enabled, RigidBody::enable_linear_motion_interpolation, and the static body
      // a static collider belongs to
      const int cf = ((d.ccd_enabled && d.ccd_enabled[k]) ? 1 : 0) |
                     ((st == NPHYS_STATUS_DYNAMIC && d.linear_motion_interpolation && d.linear_motion_interpolation[k])
                          ? 2
                          : 0);
      h_ccd.push_back(cf);
      any_ccd = any_ccd || (cf & 1) != 0;
      int ckey = n0 + k;
      if (st != NPHYS_STATUS_DYNAMIC && d.static_body && d.static_body[k] >= 0)
        ckey = static_owner.emplace(std::make_pair(h_scene.back(), int(d.static_body[k])), n0 + k).first->second;
      h_ccd_key.push_back(ckey);
      const float* p = d.pos + 3 * k;
      const float* q = d.rot + 4 * k;
      const float4 hpos = make_float4(p[0], p[1], p[2], 0.0f), hrot = make_float4(q[0], q[1], q[2], q[3]);
      hp[size_t(k) * kPoseBlock] = hpos;
      hp[size_t(k) * kPoseBlock + 1] = hrot;
      const bool dyn = st == NPHYS_STATUS_DYNAMIC;
      // ActivationStatus::new_active (body.rs:77-82): energy 4 x the default threshold 0.01
      const float thr = d.sleep_threshold ? d.sleep_threshold[k] : -1.0f;
      ha[k] = make_float2(0.01f * 4.0f, thr);
      any_sleeper = any_sleeper || (dyn && thr >= 0.0f);
      new_dynamic += dyn ? 1 : 0;
      hv[k] = (dyn && d.linvel) ? make_float4(d.linvel[3 * k], d.linvel[3 * k + 1], d.linvel[3 * k + 2], 0.0f)
                                : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      hw[k] = (dyn && d.angvel) ? make_float4(d.angvel[3 * k], d.angvel[3 * k + 1], d.angvel[3 * k + 2], 0.0f)
                                : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      // proxy creation: loose = aabb(pos) loosened by the query limit, then by 0.01
      const aabb a = shape_aabb(sh, xyz(he), xyz(hpos), toq(hrot));
      const aabb lo = loosened(loosened(a, h_qlim.back()), 0.01f);
      hmn[k] = f4(lo.mn, dyn ? 1.0f : 0.0f);
      hmx[k] = f4(lo.mx, 0.0f);
    }
    const size_t f4b = sizeof(float4);
    // grow the per-body device arrays, keeping the existing bodies' state
    for (DBuf* b : {&linvel, &angvel, &loose_mn, &loose_mx})
      HIPCK(b->ensure(size_t(n1) * f4b, true, stream));
    HIPCK(pose.ensure(size_t(n1) * kPoseBlock * f4b, true, stream));
    // kept: a sleeping body's inverse inertia is not recomputed
    HIPCK(sol.ensure(size_t(n1) * kSolverBlock * f4b, true, stream));
    HIPCK(act.ensure(size_t(n1) * sizeof(float2), true, stream));
    for (DBuf* b : {&w_dyn, &f_lin, &f_ang}) HIPCK(b->ensure(size_t(n1) * f4b, true, stream));
    for (DBuf* b : {&pos0, &rot0, &ext_lin, &ext_ang, &dims, &local_i, &damp, &surf, &rot_dyn, &groups})
      HIPCK(b->ensure(size_t(n1) * f4b));
    for (DBuf* b : {&status, &shape, &scene, &margin, &qlim, &friction, &restitution, &mass, &bflags, &matid,
                    &ccd_flags, &ccd_keys})
      HIPCK(b->ensure(size_t(n1) * 4));
    HIPCK(ccd_rot.ensure(size_t(n1) * f4b));
    // scene bits above the Morton code: the order keeps every scene in its own key range
    int max_scene = 0;
    for (int sc : h_scene) max_scene = std::max(max_scene, sc);
    scene_bits = 0;
    while ((1 << scene_bits) <= max_scene) ++scene_bits;
    auto up = [&](DBuf& b, const void* src, size_t bytes, size_t off) {
      return hipMemcpyAsync(static_cast<char*>(b.p) + off, src, bytes, hipMemcpyHostToDevice, stream);
    };
    HIPCK(up(status, h_status.data(), size_t(n1) * 4, 0));
    HIPCK(up(shape, h_shape.data(), size_t(n1) * 4, 0));
    HIPCK(up(scene, h_scene.data(), size_t(n1) * 4, 0));
    HIPCK(up(dims, h_dims.data(), size_t(n1) * f4b, 0));
    HIPCK(up(local_i, h_local_i.data(), size_t(n1) * f4b, 0));
    HIPCK(up(mass, h_mass.data(), size_t(n1) * 4, 0));
    HIPCK(up(margin, h_margin.data(), size_t(n1) * 4, 0));
    HIPCK(up(qlim, h_qlim.data(), size_t(n1) * 4, 0));
    HIPCK(up(friction, h_friction.data(), size_t(n1) * 4, 0));
    HIPCK(up(restitution, h_restitution.data(), size_t(n1) * 4, 0));
    HIPCK(up(damp, h_damp.data(), size_t(n1) * f4b, 0));
    HIPCK(up(surf, h_surf.data(), size_t(n1) * f4b, 0));
    HIPCK(up(groups, h_groups.data(), size_t(n1) * f4b, 0));
    HIPCK(up(bflags, h_flags.data(), size_t(n1) * 4, 0));
    HIPCK(up(matid, h_matid.data(), size_t(n1) * 4, 0));
    HIPCK(up(ccd_flags, h_ccd.data(), size_t(n1) * 4, 0));
    HIPCK(up(ccd_keys, h_ccd_key.data(), size_t(n1) * 4, 0));
    // new bodies: no dynamics update yet (the augmented mass is the world inertia, w = 0) and no
    // pending force
    HIPCK(hipMemsetAsync(w_dyn.as<float4>() + n0, 0, size_t(d.n) * f4b, stream));
    HIPCK(hipMemsetAsync(f_lin.as<float4>() + n0, 0, size_t(d.n) * f4b, stream));
    HIPCK(hipMemsetAsync(f_ang.as<float4>() + n0, 0, size_t(d.n) * f4b, stream));
    HIPCK(hipMemsetAsync(sol.as<float4>() + size_t(n0) * kSolverBlock, 0, size_t(d.n) * kSolverBlock * f4b, stream));
    HIPCK(hipMemcpyAsync(act.as<float2>() + n0, ha.data(), size_t(d.n) * sizeof(float2), hipMemcpyHostToDevice,
                         stream));
    HIPCK(up(pose, hp.data(), size_t(d.n) * kPoseBlock * f4b, size_t(n0) * kPoseBlock * f4b));
    HIPCK(up(linvel, hv.data(), size_t(d.n) * f4b, size_t(n0) * f4b));
    HIPCK(up(angvel, hw.data(), size_t(d.n) * f4b, size_t(n0) * f4b));
    HIPCK(up(loose_mn, hmn.data(), size_t(d.n) * f4b, size_t(n0) * f4b));
    HIPCK(up(loose_mx, hmx.data(), size_t(d.n) * f4b, size_t(n0) * f4b));
    // per-scene dynamic-body lists of the scene-blocked sweeps
    nscenes = 1;
    for (int sc : h_scene) nscenes = std::max(nscenes, sc + 1);
    std::vector<int> dstart(size_t(nscenes) + 1, 0), dlist, local(size_t(n1), -1);
    for (int i = 0; i < n1; ++i)
      if (h_status[i] == NPHYS_STATUS_DYNAMIC) ++dstart[size_t(h_scene[i]) + 1];
    max_scene_dyn = 0;
    for (int sc = 0; sc < nscenes; ++sc) {
      max_scene_dyn = std::max(max_scene_dyn, dstart[size_t(sc) + 1]);
      dstart[size_t(sc) + 1] += dstart[size_t(sc)];
    }
    dlist.resize(size_t(dstart[size_t(nscenes)]));
    {
      std::vector<int> fill(dstart.begin(), dstart.end() - 1);
      for (int i = 0; i < n1; ++i)
        if (h_status[i] == NPHYS_STATUS_DYNAMIC) {
          const int sc = h_scene[i];
          local[size_t(i)] = fill[size_t(sc)] - dstart[size_t(sc)];
          dlist[size_t(fill[size_t(sc)]++)] = i;
        }
    }
    HIPCK(sc_dyn_start.ensure(dstart.size() * 4));
    HIPCK(sc_dyn_list.ensure(std::max<size_t>(dlist.size(), 1) * 4));
    HIPCK(sc_local.ensure(local.size() * 4));
    HIPCK(up(sc_dyn_start, dstart.data(), dstart.size() * 4, 0));
    if (!dlist.empty()) HIPCK(up(sc_dyn_list, dlist.data(), dlist.size() * 4, 0));
    HIPCK(up(sc_local, local.data(), local.size() * 4, 0));
    {
      std::vector<int> small, large;
      for (int sc = 0; sc < nscenes; ++sc) {
        const int nd = dstart[size_t(sc) + 1] - dstart[size_t(sc)];
        if (nd == 0) continue;
        (nd <= kSmallScene ? small : large).push_back(sc);
      }
      n_small_scenes = int(small.size());
      n_large_scenes = int(large.size());
      HIPCK(sc_small.ensure(std::max<size_t>(small.size(), 1) * 4));
      HIPCK(sc_large.ensure(std::max<size_t>(large.size(), 1) * 4));
      if (!small.empty()) HIPCK(up(sc_small, small.data(), small.size() * 4, 0));
      if (!large.empty()) HIPCK(up(sc_large, large.data(), large.size() * 4, 0));
    }
    fixed_end = 0;
    for (int i = 0; i < n1; ++i)
      if (h_status[size_t(i)] != NPHYS_STATUS_DYNAMIC) fixed_end = i + 1;
    any_cuboid = any_ball = false;
    for (int i = 0; i < n1; ++i) {
      any_cuboid = any_cuboid || (h_shape[size_t(i)] == NPHYS_SHAPE_CUBOID && h_status[size_t(i)] == NPHYS_STATUS_DYNAMIC);
      any_ball = any_ball || h_shape[size_t(i)] == NPHYS_SHAPE_BALL;
    }
    tune_cands.clear();
    tuned = false;
    HIPCK(hipStreamSynchronize(stream));
    n = n1;
    n_dynamic += new_dynamic;
    sleeping = sleeping || any_sleeper;
    pairs_dirty = true;
    moved = true;
    return NPHYS_OK;
  }

  // At least `need` bytes of the staging buffer, which grows by half at least: contacts and pairs read at every
  // frame of a filling scene would else pin a new buffer at each.
  int io_room(size_t need) {
    if (need <= io_cap) return NPHYS_OK;
    need = std::max(need, io_cap + io_cap / 2);
    HIPCK(hipStreamSynchronize(stream));
    if (io_host) (void)hipHostFree(io_host);
    io_host = nullptr;
    io_cap = 0;
    HIPCK(hipHostMalloc(reinterpret_cast<void**>(&io_host), need, hipHostMallocMapped | hipHostMallocCoherent));
    HIPCK(hipHostGetDevicePointer(reinterpret_cast<void**>(&io_dev), io_host, 0));
    io_cap = need;
    return NPHYS_OK;
  }

  // Where the four packed state arrays stand in the pinned staging buffer (grown to fit, at 16-byte
  // aligned starts): as the host and as the device address them.
  int state_rows(const bool (&want)[4], StateRows& host, StateRows& dev) {
    const size_t pad = (size_t(n) + 3) & ~size_t(3);
    const int rc = io_room(pad * 13 * sizeof(float));
    if (rc) return rc;
    const size_t off[4] = {0, pad * 3, pad * 7, pad * 10};
    for (int a = 0; a < 4; ++a) {
      host.row[a] = want[a] ? io_host + off[a] : nullptr;
      dev.row[a] = want[a] ? io_dev + off[a] : nullptr;
    }
    return NPHYS_OK;
  }

  int set_state(const float* p, const float* r, const float* lv, const float* av) {
    if (n == 0) return NPHYS_OK;
    if (r && !rot_dyn_saved) {
      // impulses applied before the next step use the augmented mass of the rotation the last
      // dynamics update saw (the reference recomputes it only in the next step)
      launch_save_rot_dyn(bodies(), rot_dyn.as<float4>(), stream);
      rot_dyn_saved = true;
    }
    const float* in[4] = {p, r, lv, av};
    StateRows host, dev;
    int rc = state_rows({p != nullptr, r != nullptr, lv != nullptr, av != nullptr}, host, dev);
    if (rc) return rc;
    for (int a = 0; a < 4; ++a)
      if (in[a]) std::memcpy(host.row[a], in[a], size_t(n) * (a == 1 ? 4 : 3) * sizeof(float));
    launch_state_in(bodies(), dev, stream);
    if (sleeping || any_ccd) launch_clear_dyn_marks(bodies(), stream);
    if ((rc = readback({}))) return rc;  // the staging buffer has been read
    moved = true;
    wake_pending = sleeping;
    return NPHYS_OK;
  }

  int set_collision_groups(int32_t count, const int32_t* bodies_, const uint32_t* g) {
    if (count < 0 || (count > 0 && (!bodies_ || !g))) return set_err(NPHYS_ERR_INVALID, "bad collision group arrays");
    for (int k = 0; k < count; ++k)
      if (bodies_[k] < 0 || bodies_[k] >= n) return set_err(NPHYS_ERR_INVALID, "bad body handle");
    if (count == 0) return NPHYS_OK;
    constexpr uint32_t kAllGroups = (1u << 30) - 1u;
    for (int k = 0; k < count; ++k)
      h_groups[size_t(bodies_[k])] = make_uint4(g[3 * k] & kAllGroups, g[3 * k + 1] & kAllGroups, g[3 * k + 2] & kAllGroups, 0u);
    any_groups = false;
    for (const uint4& cg : h_groups) any_groups = any_groups || cg.x != kAllGroups || cg.y != kAllGroups || cg.z != 0u;
    HIPCK(hipMemcpyAsync(groups.p, h_groups.data(), size_t(n) * sizeof(uint4), hipMemcpyHostToDevice, stream));
    HIPCK(hipStreamSynchronize(stream));
    pairs_dirty = true;
    recollide = true;
    return NPHYS_OK;
  }

  int read_activation(float* energy, int64_t cap) {
    if (cap < n) return set_err(NPHYS_ERR_CAPACITY, "energy buffer too small");
    if (n == 0) return NPHYS_OK;
    std::vector<float2> h(static_cast<size_t>(n));
    HIPCK(hipMemcpyAsync(h.data(), act.p, size_t(n) * sizeof(float2), hipMemcpyDeviceToHost, stream));
    HIPCK(hipStreamSynchronize(stream));
    for (int i = 0; i < n; ++i) energy[i] = h[size_t(i)].x;
    return NPHYS_OK;
  }

  int get_state(float* p, float* r, float* lv, float* av) {
    if (n == 0) return NPHYS_OK;
    float* out[4] = {p, r, lv, av};
    StateRows host, dev;
    int rc = state_rows({p != nullptr, r != nullptr, lv != nullptr, av != nullptr}, host, dev);
    if (rc) return rc;
    launch_state_out(bodies(), dev, stream);
    if ((rc = readback({}))) return rc;
    for (int a = 0; a < 4; ++a)
      if (out[a]) std::memcpy(out[a], host.row[a], size_t(n) * (a == 1 ? 4 : 3) * sizeof(float));
    return NPHYS_OK;
  }

  // ------------------------------------------------------------------ broad phase
  int ensure_bp() {
    const size_t nn = size_t(std::max(n, 2));
    if (!direct_pairs()) {
      for (DBuf* b : {&keys, &vals, &keys_alt, &vals_alt}) HIPCK(b->ensure(nn * 4));
      for (DBuf* b : {&leaf_mn, &leaf_mx}) HIPCK(b->ensure(nn * sizeof(float4)));
      for (DBuf* b : {&box_mn, &box_mx}) HIPCK(b->ensure(search_boxes(nn) * sizeof(float4)));
      HIPCK(box_top.ensure(search_boxes(nn) * 4));
      HIPCK(bp_tmp.ensure(radix_temp_words(int(nn)) * 4));
      HIPCK(scan.ensure(radix_scan_tiles(int(nn)), stream));
    }
    HIPCK(cand_count.ensure(nn * 4));
    if (cand.bytes < nn * size_t(cap) * 4) segments_valid = false;  // segments are lost on growth
    HIPCK(cand.ensure(nn * size_t(cap) * 4));
    HIPCK(bp_list.ensure(nn * 4));
    if (bp_dirty.bytes < nn * 4) {
      segments_valid = false;
      HIPCK(bp_dirty.ensure(nn * 4));
      fill_u32(bp_dirty.as<uint32_t>(), 0u, nn, stream);
    }
    HIPCK(scan.ensure(compact_tiles(int(nn)), stream));
    return NPHYS_OK;
  }

  // Whether the pair search does without the order and its boxes (k_broadphase.hip).
  bool direct_pairs() const { return nscenes == 1 && n <= kDirectBodies; }

  BroadPhaseBufs bp_view() {
    BroadPhaseBufs v;
    uint32_t* sm = bp_small.as<uint32_t>();
    v.changed = sm;
    v.bounds = sm + 8;
    v.stats = sm + 16;
    v.keys = keys.as<uint32_t>();
    v.vals = vals.as<uint32_t>();
    v.keys_alt = keys_alt.as<uint32_t>();
    v.vals_alt = vals_alt.as<uint32_t>();
    v.leaf_mn = leaf_mn.as<float4>();
    v.leaf_mx = leaf_mx.as<float4>();
    v.box_mn = box_mn.as<float4>();
    v.box_mx = box_mx.as<float4>();
    v.box_top = box_top.as<int>();
    v.scene_bits = scene_bits;
    v.cand = cand.as<int>();
    v.cand_count = cand_count.as<uint32_t>();
    v.pairs = pairs.as<int2>();
    v.tmp = bp_tmp.as<uint32_t>();
    v.scan = &scan;
    v.dirty = bp_dirty.as<uint32_t>();
    v.list = bp_list.as<int>();
    v.list_count = sm + kSmListCount;
    return v;
  }

  // Enqueues a readback of up to four device word ranges into rb_host; returns its sequence number.
  uint32_t rb_post(std::initializer_list<RbSeg> segs) {
    RbJob j{};
    int k = 0;
    for (const RbSeg& s : segs) {
      j.src[k] = s.src;
      j.n[k] = s.n;
      j.dst[k] = s.dst;
      ++k;
    }
    ++rb_seq;
    hipLaunchKernelGGL(k_readback, dim3(1), dim3(256), 0, stream, j, rb_dev, kRbFlag, rb_seq);
    return rb_seq;
  }

  // Waits until readback `seq` (and everything before it on the stream) has completed. After two
  // seconds the stream is synchronised instead, which reports a failed launch or fault.
  int rb_wait(uint32_t seq) {
    const volatile uint32_t* f = rb_host + kRbFlag;
    const auto t0 = std::chrono::steady_clock::now();
    for (uint32_t it = 1; int32_t(*f - seq) < 0; ++it) {
      if ((it & 0xfffu) == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::seconds(2)) {
        HIPCK(hipStreamSynchronize(stream));
        if (int32_t(*f - seq) >= 0) break;
        return set_err(NPHYS_ERR_HIP, "readback did not complete");
      }
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return NPHYS_OK;
  }

  int readback(std::initializer_list<RbSeg> segs) { return rb_wait(rb_post(segs)); }

  // Words of bp_small that a detection reads back in one piece: the loose passes' counts (0-3) and the dirty
  // list's length; then what every search starts from zeroed, its largest segment, the narrow phase's contacts and
  // manifolds and the lengths of its two lists; and the pairs.
  static constexpr int kSmListCount = 4, kSmStats = 16, kSmTotals = 24, kSmBoxes = 26, kSmBalls = 27, kSmPairs = 28;

  // GeometricalWorld::sync_colliders (the loose-AABB passes of `passes`), perform_broad_phase and,
  // when `narrow`, perform_narrow_phase into cb[cur]. *changed: loose AABBs replaced. bp_done and np_done, when
  // given, are recorded after the two phases. Where it fails there are no manifolds, and no pairs unless their
  // list is complete (too many of them for the narrow phase); the next step begins with another detection.
  int detect(int passes, bool narrow, int64_t* changed, hipEvent_t bp_done = nullptr, hipEvent_t np_done = nullptr) {
    bool listed = false;
    const int rc = find_pairs(passes, narrow, changed, bp_done, np_done, listed);
    segments_valid = listed;
    pairs_dirty = !listed;
    if (!listed) npairs = 0;
    int& run = calm[narrow ? 1 : 0];
    run = rc == NPHYS_OK && *changed == 0 ? std::min(run + 1, kCalm) : 0;
    if (rc) {
      list_room = 0;
      cb[cur].C = cb[cur].M = 0;
      recollide = true;
    }
    return rc;
  }

  // Everything is enqueued with room for an eighth more pairs than last time and read back once at the end;
  // if the pairs or a body's segment did not fit, buffers grow and the launches after the loose passes
  // run again. npairs is the new list's length from when it is stored (`listed`).
  int find_pairs(int passes, bool narrow, int64_t* changed, hipEvent_t bp_done, hipEvent_t np_done, bool& listed) {
    int rc = ensure_bp();
    if (rc) return rc;
    const DevBodies b = bodies();
    BroadPhaseBufs v = bp_view();
    uint32_t* sm = bp_small.as<uint32_t>();
    const uint32_t* h = rb_host;
    // After kCalm detections in a row that replaced no loose AABB, as in a world at rest, this one is taken
    // for such a one too: the pairs and the narrow phase's lists stand, so the narrow phase follows the loose passes at once,
    // and only where the readback tells of a replaced AABB is everything searched. Broad phase at rest
    // 137 -> 16 us at 262,144 balls and 67 -> 14 at 99,996 (with a readback before every search, as there was once,
    // 22 at rest, and the search waits for it otherwise).
    const bool stand = calm[narrow ? 1 : 0] == kCalm && segments_valid && !pairs_dirty &&
                       (!narrow || (list_room > 0 && npairs <= most_pairs));
    fill_u32(sm, 0u, stand ? kSmBoxes : kSmPairs + 1, stream);
    launch_loose_update(b, passes, v, stream);
    if (stand) {
      ContactBufs& out = cb[cur];
      if (narrow) {
        NarrowPhaseBufs np{};
        if ((rc = ensure_narrow(list_room, &out, np))) return rc;
        fill_u32(out.bfirst.as<uint32_t>(), 0xffffffffu, size_t(n), stream);
        if (bp_done) HIPCK(hipEventRecord(bp_done, stream));
        launch_narrow_phase(b, pairs.as<int2>(), np, out.view(), stream);
        if (np_done) HIPCK(hipEventRecord(np_done, stream));
      }
      if ((rc = readback({{sm, kSmPairs + 1, 0}}))) return rc;
      *changed = int64_t(h[0]) + h[2];
      if (*changed == 0) {
        listed = true;
        out.C = narrow ? int(h[kSmTotals]) : out.C;
        out.M = narrow ? int(h[kSmTotals + 1]) : out.M;
        return NPHYS_OK;
      }
      fill_u32(sm + kSmStats, 0u, kSmPairs - kSmStats, stream);
    }
    const bool direct = direct_pairs();
    if (!direct && (pairs_dirty || (passes & LOOSE_STATIC) || ++order_age > kOrderAge)) {
      launch_order(b, v, stream);
      order_age = 0;
    }
    bool may = segments_valid && incremental_bp && !pairs_dirty;
    bool manifolds = narrow;
    for (int64_t want = int64_t(npairs) + npairs / 8 + 1024;;) {
      const int room = int(std::min<int64_t>(want, manifolds ? most_pairs : INT_MAX));
      ContactBufs& out = cb[cur];
      NarrowPhaseBufs np{};
      if ((rc = ensure_narrow(room, manifolds ? &out : nullptr, np))) return rc;
      HIPCK(pairs.ensure(size_t(room) * sizeof(int2)));
      v = bp_view();
      SearchRun r{};
      r.direct = direct ? 1 : 0;
      r.fixed_end = fixed_end;
      r.cap = cap;
      r.may_increment = may ? 1 : 0;
      launch_search(b, v, r, stream);
      PairOut po;
      po.npairs = sm + kSmPairs;
      po.nbox = np.nbox;
      po.nball = np.nball;
      po.perm = np.perm;
      po.bfirst = manifolds ? out.bfirst.as<int>() : nullptr;
      po.pair_cap = room;
      launch_compact_pairs(b, v, cap, direct, po, stream);
      if (bp_done) HIPCK(hipEventRecord(bp_done, stream));
      if (manifolds) launch_narrow_phase(b, pairs.as<int2>(), np, out.view(), stream);
      if (np_done) HIPCK(hipEventRecord(np_done, stream));
      if ((rc = readback({{sm, kSmPairs + 1, 0}}))) return rc;
      *changed = int64_t(h[0]) + h[2];
      // the device's rule (search_incremental), for the counters
      const bool incremental = may && h[1] + h[3] == 0 && *changed <= kept_limit(n);
      if (int(h[kSmStats]) > cap) {
        // a segment took more partners than it has room for: all search again, with larger segments
        if (incremental) ++counters.incremental_overflows;
        cap = int(h[kSmStats]) + 8;
        if ((rc = ensure_bp())) return rc;
        may = false;
        fill_u32(sm + kSmStats, 0u, kSmPairs - kSmStats, stream);
        continue;
      }
      const uint32_t found = h[kSmPairs];
      if (found > uint32_t(room)) {
        if (found > uint32_t(INT_MAX)) return set_err(NPHYS_ERR_CAPACITY, "too many broad-phase pairs");
        manifolds = manifolds && int(found) <= most_pairs;  // else the pair list alone
        want = int64_t(found) + found / 8;
        // the segments stand, and as the dirty flags are cleared an incremental search keeps them
        fill_u32(sm + kSmStats, 0u, kSmPairs - kSmStats, stream);
        continue;
      }
      npairs = int(found);
      listed = true;
      list_room = room;
      if (incremental && *changed != 0) ++counters.incremental_pair_updates;
      if (!narrow) return NPHYS_OK;
      if (!manifolds) return set_err(NPHYS_ERR_CAPACITY, "too many broad-phase pairs");
      out.C = int(h[kSmTotals]);
      out.M = int(h[kSmTotals + 1]);
      return NPHYS_OK;
    }
  }

  int pairs_out(int32_t* out) {
    const size_t bytes = size_t(npairs) * sizeof(int2);
    int rc = io_room(bytes);
    if (rc) return rc;
    HIPCK(hipMemcpyAsync(io_host, pairs.p, bytes, hipMemcpyDeviceToHost, stream));
    HIPCK(hipStreamSynchronize(stream));
    std::memcpy(out, io_host, bytes);
    return NPHYS_OK;
  }

  // The contacts of `c` in manifold order into `out` (arrays may be null): their places by a prefix sum, the
  // arrays written by the device in the staging buffer.
  int contacts_out(ContactBufs& c, const ContactRows& out) {
    const int M = c.M;
    const size_t C = size_t(c.C), pad = (C + 3) & ~size_t(3);
    HIPCK(rd_moff.ensure(size_t(std::max(M, 1)) * 4));
    HIPCK(scan.ensure(scan_tiles(size_t(std::max(M, 1))), stream));
    int rc = io_room((pad * 13 + 4) * sizeof(float));
    if (rc) return rc;
    ContactRows dev, host;
    size_t off = 4;  // the first word: the contacts counted
    for (int a = 0; a < ContactRows::kRows; ++a) {
      host.row[a] = io_host + off;
      dev.row[a] = out.row[a] ? io_dev + off : nullptr;
      off += pad * ContactRows::kWidth[a];
    }
    const DevContacts v = c.view();
    scan_exclusive_u32(reinterpret_cast<const uint32_t*>(v.mcount), rd_moff.as<uint32_t>(), M, scan, stream);
    launch_contacts_out(v, M, rd_moff.as<uint32_t>(), uint32_t(C), dev, reinterpret_cast<uint32_t*>(io_dev), stream);
    if ((rc = readback({}))) return rc;
    uint32_t counted;
    std::memcpy(&counted, io_host, 4);
    if (counted != uint32_t(C)) return set_err(NPHYS_ERR_STATE, "contact count mismatch");
    for (int a = 0; a < ContactRows::kRows; ++a)
      if (out.row[a]) std::memcpy(out.row[a], host.row[a], C * size_t(ContactRows::kWidth[a]) * sizeof(float));
    return NPHYS_OK;
  }

  // The contacts of `c` in manifold order (dense records and, when imp is given, impulses), with
  // the manifolds' bodies and counts, copied to the host.
  int gather_contacts(ContactBufs& c, std::vector<int2>& mb, std::vector<int>& mc, std::vector<float4>& rec,
                      std::vector<float4>* imp) {
    const int M = c.M, C = c.C;
    mb.resize(size_t(M));
    mc.resize(size_t(M));
    HIPCK(hipMemcpyAsync(mb.data(), c.mbody.p, size_t(M) * sizeof(int2), hipMemcpyDeviceToHost, stream));
    HIPCK(hipMemcpyAsync(mc.data(), c.mcount.p, size_t(M) * 4, hipMemcpyDeviceToHost, stream));
    HIPCK(hipStreamSynchronize(stream));
    std::vector<uint32_t> off(static_cast<size_t>(M));
    uint32_t acc = 0;
    for (int m = 0; m < M; ++m) {
      off[size_t(m)] = acc;
      acc += uint32_t(mc[size_t(m)]);
    }
    if (int(acc) != C) return set_err(NPHYS_ERR_STATE, "contact count mismatch");
    HIPCK(rd_moff.ensure(size_t(std::max(M, 1)) * 4));
    HIPCK(rd_rec.ensure(size_t(std::max(C, 1)) * kContactFields * sizeof(float4)));
    if (imp) HIPCK(rd_imp.ensure(size_t(std::max(C, 1)) * sizeof(float4)));
    HIPCK(hipMemcpyAsync(rd_moff.p, off.data(), size_t(M) * 4, hipMemcpyHostToDevice, stream));
    launch_gather_contacts(c.view(), M, rd_moff.as<uint32_t>(), rd_rec.as<float4>(),
                           imp ? rd_imp.as<float4>() : nullptr, stream);
    rec.resize(size_t(C) * kContactFields);
    HIPCK(hipMemcpyAsync(rec.data(), rd_rec.p, rec.size() * sizeof(float4), hipMemcpyDeviceToHost, stream));
    if (imp) {
      imp->resize(size_t(C));
      HIPCK(hipMemcpyAsync(imp->data(), rd_imp.p, imp->size() * sizeof(float4), hipMemcpyDeviceToHost, stream));
    }
    HIPCK(hipStreamSynchronize(stream));
    return NPHYS_OK;
  }

  // ------------------------------------------------------------------ narrow phase
  // Buffers of a narrow phase over `room` pairs (and its output's, when given); `v` describes them.
  int ensure_narrow(int room, ContactBufs* out, NarrowPhaseBufs& v) {
    const size_t P = size_t(std::max(room, 1));
    for (DBuf* b : {&np_count, &np_perm}) HIPCK(b->ensure(P * 4));
    HIPCK(scan.ensure(manifold_tiles(int(P)), stream));
    if (out) {
      HIPCK(out->ensure(P, kPairSlots * P));
      HIPCK(out->bfirst.ensure(size_t(std::max(n, 1)) * 4));
      out->nb = n;
    }
    uint32_t* sm = bp_small.as<uint32_t>();
    v.count = np_count.as<uint32_t>();
    v.perm = np_perm.as<uint32_t>();
    v.npairs = sm + kSmPairs;
    v.nbox = sm + kSmBoxes;
    v.nball = sm + kSmBalls;
    v.totals = sm + kSmTotals;
    v.pair_cap = int(P);
    v.boxes = any_cuboid;
    v.balls = any_ball;
    v.scan = &scan;
    return NPHYS_OK;
  }

  // The narrow phase of `np` pairs (in pair order; their number also at *count_dev) into `out`. Without
  // `totals`, the host does not wait for its contact and manifold counts.
  int narrow_phase_of(const int2* list, int np, uint32_t* count_dev, ContactBufs& out, bool totals = true) {
    if (np > most_pairs) return set_err(NPHYS_ERR_CAPACITY, "too many broad-phase pairs");
    NarrowPhaseBufs v{};
    list_room = 0;  // the lists become those of `list`
    const int rc0 = ensure_narrow(np, &out, v);
    if (rc0) return rc0;
    v.npairs = count_dev;
    fill_u32(v.totals, 0u, 4, stream);
    launch_narrow_bins(bodies(), list, v, out.view(), stream);
    launch_narrow_phase(bodies(), list, v, out.view(), stream);
    if (!totals) return NPHYS_OK;
    const int rc = readback({{v.totals, 2, 0}});
    if (rc) return rc;
    out.C = int(rb_host[0]);
    out.M = int(rb_host[1]);
    return NPHYS_OK;
  }

  // Collision detection on the current poses of every body, static ones included.
  int collide_now() {
    int64_t changed = 0;
    return detect(LOOSE_FINAL | LOOSE_STATIC, true, &changed);
  }

  // ------------------------------------------------------------------ solver
  // Whether this solve computes the network's features, which tell cached impulses from new ones.
  bool learned_rows() const { return capture || contact_model == NPHYS_CONTACT_MODEL_LEARNED_WARMSTART; }

  int ensure_solver(int M, int C, int digits = kColourDigits) {
    const size_t nn = size_t(std::max(n, 1));
    const size_t m = size_t(std::max(M, 1)), c = size_t(std::max(C, 1));
    for (DBuf* b : {&sv_deg, &sv_adj_off}) HIPCK(b->ensure(nn * 4));
    HIPCK(sv_adj.ensure(2 * m * 4));
    HIPCK(sv_place.ensure(m * sizeof(uint2)));
    HIPCK(sv_ckeys.ensure(m * 4));
    HIPCK(sv_slot_of.ensure(m * sizeof(uint2)));
    HIPCK(sv_state2[cur].ensure(m * 4));
    HIPCK(sv_state2[cur ^ 1].ensure(4));
    HIPCK(sv_col_start.ensure(2 * (kMaxColours + 2) * 4));
    const size_t hw = colour_hist_words(int(m), digits);
    HIPCK(sv_hist.ensure(2 * hw * 4));
    HIPCK(sv_sinfo.ensure(m * sizeof(int4)));
    HIPCK(sv_rec.ensure(c * kRecFields * sizeof(float4)));
    HIPCK(sv_lam.ensure(c * sizeof(float4)));
    if (learned_rows()) HIPCK(sv_has.ensure(c * 4));
    HIPCK(sv_prec.ensure(c * 3 * sizeof(float4)));
    HIPCK(sv_pgeo.ensure(m * 2 * sizeof(float4)));
    rec_stride = long(std::min({sv_rec.bytes / (kRecFields * sizeof(float4)), sv_lam.bytes / sizeof(float4),
                                sv_prec.bytes / (3 * sizeof(float4))}));
    HIPCK(scan.ensure(std::max(scan_tiles(hw), scan_tiles(nn)), stream));
    return NPHYS_OK;
  }

  SolverBufs sv_view() {
    SolverBufs v;
    v.deg = sv_deg.as<uint32_t>();
    v.adj_off = sv_adj_off.as<uint32_t>();
    v.adj = sv_adj.as<int>();
    v.place = sv_place.as<uint2>();
    v.state = sv_state2[cur].as<uint32_t>();
    v.hist = sv_hist.as<uint32_t>();
    v.offs = v.hist + sv_hist.bytes / 8;
    v.ckeys = sv_ckeys.as<uint32_t>();
    v.col_start = sv_col_start.as<uint32_t>();
    v.class_rec = v.col_start + (kMaxColours + 2);
    v.sinfo = sv_sinfo.as<int4>();
    v.slot_of = sv_slot_of.as<uint2>();
    v.rec_stride = rec_stride;
    v.rec = sv_rec.as<float4>();
    v.lam = sv_lam.as<float4>();
    v.prec = sv_prec.as<float4>();
    v.pgeo = sv_pgeo.as<float4>();
    v.red = red_dev;
    v.has = learned_rows() ? sv_has.as<float>() : nullptr;
    v.tmp = sv_tmp.as<uint32_t>();
    v.scan = &scan;
    return v;
  }

  // Visit order of the colour classes for one solve: Fisher-Yates driven by SplitMix64 seeded
  // with the solve index, so every step orders conflicting manifolds afresh while the colours
  // themselves persist between steps; then stably sorted by size bucket floor(log2(size)),
  // smallest first, so the largest classes end every sweep (the rows solved last are the most
  // numerous: a lower residual at equal iteration count).
  static int size_bucket(int n) {
    int l = 0;
    while (l < 30 && (2 << l) <= n) ++l;
    return l;
  }
  static void colour_visit_order(uint64_t solve_index, int k, const int* size, std::vector<int>& perm) {
    perm.resize(k);
    for (int c = 0; c < k; ++c) perm[c] = c;
    uint64_t st = solve_index * 0x9E3779B97F4A7C15ull;
    for (int i = k - 1; i > 0; --i) {
      st += 0x9E3779B97F4A7C15ull;
      uint64_t z = st;
      z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
      z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
      z ^= z >> 31;
      const int j = int(z % uint64_t(i + 1));
      std::swap(perm[i], perm[j]);
    }
    std::stable_sort(perm.begin(), perm.end(), [&](int a, int b) { return size_bucket(size[a]) < size_bucket(size[b]); });
  }

  // Words of bp_small of the colouring: whether a round of a batch but the last, and the last one, left a
  // manifold uncoloured, the number of colours, the last round that coloured one.
  static constexpr int kSmRemaining = 32, kSmColours = kSmRemaining + 2, kSmLastRound = kSmColours + 1, kSmColouring = 4;

  // Colouring, slots and assembly of the solve's manifolds, and the class bounds back on the host
  // (colour_visit, h_span, class_contacts). The rounds run in batches: a round after the last one that
  // colours anything changes nothing, and the device records that last round. A batch, the colour order and the assembly
  // are enqueued together and read back once; where manifolds stay uncoloured, or there are more
  // colours than the order has digits for, the rest runs again. `after` enqueues what does not depend on the colouring, before the wait.
  template <class F>
  int colour_and_assemble(const DevBodies& b, const DevContacts& c, int M, int C, const SimParams& ps, SolverBufs& v,
                          F&& after) {
    // colours are inherited from the manifolds of the previous solve
    const int prevM = have_solved ? sview_M[cur ^ 1] : 0;
    const ContactBufs& pc = cb[cur ^ 1];
    uint32_t* sm = bp_small.as<uint32_t>();
    const uint32_t* prev_state = sv_state2[cur ^ 1].as<uint32_t>();
    int digits = kColourDigits;
    // recorded samples and predictions keep the row order that does not depend on the contact counts
    split_order = !learned_rows();
    // one workgroup while its lanes have two manifolds each at most (as many as its LDS holds with the bodies, and a
    // world whose launches cost more than they do), and not soon after one that was too crowded for it
    int& wait_small = crowded[ccd_sub ? 1 : 0];
    const bool small = M <= kSmallManifolds && n <= kSmallColourBodies && wait_small == 0;
    if (wait_small > 0) --wait_small;
    if (small) launch_colour_small(b, c, M, C, sview[cur ^ 1], prevM, prev_state, split_order, v, sm + kSmRemaining, stream);
    else launch_colour_begin(b, c, M, sview[cur ^ 1], prevM, prev_state, v, stream);
    bool rounds = !small, ordered = small, waiting = true;
    int& batch = round_batch[ccd_sub ? 1 : 0];
    for (int round = 1;;) {
      if (rounds) {
        if (round + batch >= 0xffff) return set_err(NPHYS_ERR_STATE, "colouring did not converge");
        // the last round's word stays when this is not the first batch
        fill_u32(sm + kSmRemaining, 0u, round == 1 ? kSmColouring : kSmColouring - 1, stream);
        for (int k = 0; k < batch; ++k, ++round)
          launch_colour_round(c, M, round, sm + kSmRemaining + (k == batch - 1 ? 1 : 0), sm + kSmLastRound, v, stream);
      }
      if (!ordered) launch_colour_order(c, M, C, digits, split_order, v, sm + kSmColours, stream);
      ordered = false;
      const uint32_t seq = rb_post({{sm + kSmRemaining, kSmColouring, 0},
                                    {v.col_start, digits + 1, kRbClass},
                                    {v.class_rec, digits + 1, kRbClass + kMaxColours + 2}});
      launch_assemble(b, c, pc.view(), have_solved ? pc.M : 0, M, ps, v, mat_table(), stream);
      if (waiting) after();
      waiting = false;
      const int rc = rb_wait(seq);
      if (rc) return rc;
      rounds = rb_host[1] != 0;
      if (small && rounds && round == 1) wait_small = kCrowdedSolves;
      ncolours = int(rb_host[kSmColours - kSmRemaining]);
      if (rounds) continue;
      if (ncolours > kMaxColours) return set_err(NPHYS_ERR_STATE, "too many colours");
      if (ncolours * (split_order ? 2 : 1) <= digits) break;
      digits = kMaxColours;
      split_order = false;
      const int rc2 = ensure_solver(M, C, digits);
      if (rc2) return rc2;
      v = sv_view();
    }
    colour_rounds = int(rb_host[kSmLastRound - kSmRemaining]);
    if (colour_rounds > 0 || !small) batch = std::min(std::max(colour_rounds + 1, kMinRounds), kMaxRounds);
    // visit order (the SplitMix64 Fisher-Yates shuffle seeded by the solve index), slot ranges in that
    // order and the largest class
    const uint32_t* h_colstart = rb_host + kRbClass;
    const uint32_t* h_rec = h_colstart + kMaxColours + 2;
    const int per = split_order ? 2 : 1;
    int csize[kMaxColours];
    for (int k = 0; k < ncolours; ++k) csize[k] = int(h_colstart[per * (k + 1)] - h_colstart[per * k]);
    colour_visit_order(uint64_t(solve_count), ncolours, csize, colour_visit);
    h_span.resize(size_t(ncolours));
    class_contacts.resize(size_t(ncolours));
    for (int k = 0; k < ncolours; ++k) {
      const int col = colour_visit[size_t(k)];
      ClassSpan& r = h_span[size_t(k)];
      r.first = int(h_colstart[per * col]);
      r.multi = int(h_colstart[per * col + 1]) - r.first;
      r.single = csize[col] - r.multi;
      class_contacts[size_t(k)] = int(h_rec[per * (col + 1)] - h_rec[per * col]);
    }
    return NPHYS_OK;
  }

  static int run_lanes(const ClassSpan& c) { return 8 * c.multi + 2 * c.single; }
  // The run of small classes that starts with the k-th visited one (at most kRunClasses of them).
  ClassRun small_run(int k, int ncol) const {
    ClassRun run;
    run.n = 0;
    for (; k < ncol && run.n < kRunClasses && run_lanes(h_span[size_t(k)]) <= kRunLanes; ++k)
      run.r[run.n++] = h_span[size_t(k)];
    return run;
  }

  VisitOrder visit_list() const {
    VisitOrder v;
    v.n = ncolours;
    v.split = split_order ? 1 : 0;
    for (int k = 0; k < ncolours; ++k) v.c[k] = uint16_t(colour_visit[size_t(k)]);
    return v;
  }

  // Warm start (when `warm`) and `nsweeps` coloured SOR-Prox sweeps. With counters enabled the
  // per-colour sweep kernels carry HIP events in their dispatch packets. Every launch is direct:
  // one per colour class, or one workgroup for a run of consecutive small classes.
  int sweeps(const DevBodies& b, SolverBufs& v, bool warm, int nsweeps) {
    if (cur_variant > 0) {
      // scene-blocked: one launch for the warm start and all nsweeps sweeps
      SceneBlocks sc = sc_view();
      if (counters_enabled) {
        while (kt_ev.size() < size_t(kt_used) + 2) {
          hipEvent_t e;
          HIPCK(hipEventCreate(&e));
          kt_ev.push_back(e);
        }
        HIPCK(hipEventRecord(kt_ev[kt_used], stream));
      }
      HIPCK(hipEventRecord(fork_ev, stream));
      HIPCK(hipStreamWaitEvent(stream_large, fork_ev, 0));
      launch_sweeps_blocked(b, v, sc, visit_list(), nsweeps, warm, cur_variant, stream, stream_large);
      HIPCK(hipEventRecord(join_ev, stream_large));
      HIPCK(hipStreamWaitEvent(stream, join_ev, 0));
      if (counters_enabled) {
        HIPCK(hipEventRecord(kt_ev[kt_used + 1], stream));
        kt_used += 2;
      }
      return NPHYS_OK;
    }
    // Direct launches (the visiting order changes every solve, so the launch sequence does): two or
    // more consecutive small classes of the visiting order run back to back in one workgroup. With
    // counters enabled each k_pgs launch carries HIP events in its dispatch packet.
    if (counters_enabled) {
      const size_t need = size_t(kt_used) + size_t(2) * size_t(nsweeps) * size_t(ncolours);
      while (kt_ev.size() < need) {
        hipEvent_t e;
        HIPCK(hipEventCreate(&e));
        kt_ev.push_back(e);
      }
    }
    auto pass = [&](bool w) {
      for (int k = 0; k < ncolours;) {
        const ClassRun run = small_run(k, ncolours);
        if (run.n >= 2) {
          launch_colour_run(b, v, run, w, stream);
          k += run.n;
          continue;
        }
        const ClassSpan& r = h_span[size_t(k)];
        if (w) {
          launch_warmstart_colour(b, r, v, stream);
        } else if (counters_enabled) {
          launch_pgs_colour(b, r, v, stream, kt_ev[kt_used], kt_ev[kt_used + 1]);
          kt_used += 2;
          counters.sweep_kernel_contacts += class_contacts[size_t(k)];
        } else {
          launch_pgs_colour(b, r, v, stream);
        }
        ++k;
      }
    };
    // the joints' rows: warm-started after the contacts' (sor_prox.rs:56-58), solved before the
    // contacts' in every sweep (sor_prox.rs:167-168)
    JointBufs jv = joint_view();
    const bool joints = nj > 0 && !ccd_sub;  // a CCD substep solves no joints (mechanical_world.rs:909)
    if (warm) {
      pass(true);
      if (joints) launch_joint_warm(b, jv, stream);
    }
    for (int it = 0; it < nsweeps; ++it) {
      if (joints) launch_joint_sweep(b, jv, stream);
      pass(false);
    }
    return NPHYS_OK;
  }

  // Natural-map residual of the current impulses: the per-block partials go straight to host memory and
  // are reduced there in block order (max is exact; the sum of squares is the RMS) once the stream
  // has passed them: residual() waits, while the fixed-count mode's, which nothing in the step
  // needs, is reduced after the step's last readback (with `cache` the kernel stores the impulses too). The
  // buffer grows here alone: a CCD substep, which solves in between, has no residual.
  int residual_deferred(const DevBodies& b, const DevContacts& cv, int M, int C, bool cache, SolverBufs& v) {
    const int nbk = residual_blocks(M);
    const size_t need = size_t(nbk) * 2 + 4;  // + the joints' partial
    if (need > red_cap) {
      HIPCK(hipStreamSynchronize(stream));
      if (red_host) (void)hipHostFree(red_host);
      red_host = nullptr;
      red_cap = 0;
      const size_t grown = std::max<size_t>(need + need / 2, 1024);
      HIPCK(hipHostMalloc(reinterpret_cast<void**>(&red_host), grown * sizeof(double),
                          hipHostMallocMapped | hipHostMallocCoherent));
      red_cap = grown;
      HIPCK(hipHostGetDevicePointer(reinterpret_cast<void**>(&red_dev), red_host, 0));
    }
    v.red = red_dev;
    launch_residual(b, cv, M, cache, v, stream);
    JointBufs jv = joint_view();
    if (nj > 0) launch_joint_residual(b, jv, v.red + 2 * nbk, stream);
    res_pending_blocks = nbk;
    res_pending_C = C;
    res_pending_joints = nj > 0;
    return NPHYS_OK;
  }
  bool res_pending_joints = false;

  void finish_residual() {
    if (res_pending_blocks < 0) return;
    double mx = 0.0, ss = 0.0, rows = double(3 * res_pending_C);
    for (int k = 0; k < res_pending_blocks; ++k) {
      mx = std::max(mx, red_host[2 * k]);
      ss += red_host[2 * k + 1];
    }
    if (res_pending_joints) {  // the joint rows' partial after the contacts' blocks
      const double* jp = red_host + 2 * res_pending_blocks;
      mx = std::max(mx, jp[0]);
      ss += jp[1];
      rows += jp[2];
    }
    res_inf = mx;
    res_rms = rows > 0.0 ? std::sqrt(ss / rows) : 0.0;
    res_pending_blocks = -1;
  }

  int residual(const DevBodies& b, const DevContacts& cv, int M, int C, SolverBufs& v) {
    int rc = residual_deferred(b, cv, M, C, false, v);
    if (rc || (rc = readback({}))) return rc;
    finish_residual();
    return NPHYS_OK;
  }

  SceneBlocks sc_view() {
    SceneBlocks v;
    v.keys = sc_keys.as<uint32_t>();
    v.slot = nscenes > 1 ? sc_slot.as<uint32_t>() : nullptr;
    v.keys_alt = sc_keys_alt.as<uint32_t>();
    v.slot_alt = sc_slot_alt.as<uint32_t>();
    v.start = nscenes > 1 ? sc_start.as<uint32_t>() : sv_col_start.as<uint32_t>();
    v.info = sc_info.as<int4>();
    v.rank = sc_rank.as<int2>();
    v.dyn_start = sc_dyn_start.as<int>();
    v.dyn_list = sc_dyn_list.as<int>();
    v.local = sc_local.as<int>();
    v.small_list = sc_small.as<int>();
    v.large_list = sc_large.as<int>();
    v.n_small = n_small_scenes;
    v.n_large = n_large_scenes;
    return v;
  }

  // One colour takes as many launches as there are sweeps, each on the whole chip (53 us a solve of 1,900 boxes on a
  // ground, 1,138 in a workgroup of 256 lanes), so there the variant is not obeyed.
  bool blocked_eligible(int ncol) const {
    return max_scene_dyn <= kLdsBodies && ncol >= 2 && ncol <= kVisitColours &&
           int64_t(nscenes) * (2 * ncol + 1) <= (int64_t(1) << 25);
  }

  // Variant of this solve's sweeps: forced, or the autotuner's pick, or (while tuning) the next
  // candidate to time. All variants give identical results.
  void choose_variant(int M) {
    tune_pending = false;
    // the scene-blocked kernels solve contacts only: worlds with joints use per-colour launches
    if (nj > 0 || !blocked_eligible(ncolours)) {
      cur_variant = 0;
      return;
    }
    if (variant_request >= 0) {
      cur_variant = variant_request;
      return;
    }
    // a pick is kept while the problem stays of the size it was timed at (a batch of falling
    // scenes has few manifolds at first): retime when the manifold count leaves [2/3, 3/2] of it
    if (tuned && (2 * int64_t(M) > 3 * int64_t(tune_M) || 3 * int64_t(M) < 2 * int64_t(tune_M))) {
      tune_cands.clear();
      tuned = false;
    }
    if (tune_cands.empty()) {
      tune_M = M;
      tune_cands = {0, 256, 512, 1024};
      tune_time.assign(tune_cands.size(), 0.0);
      tune_count.assign(tune_cands.size(), 0);
    }
    if (!tuned) {
      size_t k = 0;
      while (k < tune_cands.size() && tune_count[k] >= kTuneReps) ++k;
      if (k < tune_cands.size()) {
        cur_variant = tune_cands[k];
        tune_pending = true;
        return;
      }
      size_t best = 0;
      for (size_t i = 1; i < tune_cands.size(); ++i)
        if (tune_time[i] < tune_time[best]) best = i;
      cur_variant = tune_cands[best];
      tuned = true;
    }
  }

  void tune_record() {
    if (!tune_pending) return;
    float ms = 0.0f;
    if (hipEventElapsedTime(&ms, tune_ev[0], tune_ev[1]) != hipSuccess) return;
    for (size_t i = 0; i < tune_cands.size(); ++i)
      if (tune_cands[i] == cur_variant) {
        tune_time[i] += double(ms);
        ++tune_count[i];
      }
    tune_pending = false;
  }

  // Warm start and SOR-Prox sweeps: the fixed count of the reference (sor_prox.rs:56-79), or, in
  // solve-to-residual mode, sweeps until max |phi| <= res_target, checked after the warm start
  // and every res_check_every sweeps, at most res_max_sweeps. Leaves the final residual in
  // res_inf / res_rms and the sweep count in nsw.
  int solve_sweeps(const DevBodies& b, const DevContacts& cv, SolverBufs& v, int M, int C, int& nsw) {
    int rc;
    if (res_target <= 0.0) {
      if ((rc = sweeps(b, v, true, prm.max_velocity_iterations))) return rc;
      nsw = prm.max_velocity_iterations;
      return residual_deferred(b, cv, M, C, true, v);
    }
    if ((rc = sweeps(b, v, true, 0))) return rc;
    int done = 0;
    for (;;) {
      if ((rc = residual(b, cv, M, C, v))) return rc;
      if ((res_norm == NPHYS_RESIDUAL_RMS ? res_rms : res_inf) <= res_target || done >= res_max_sweeps) break;
      const int k = std::min(res_check_every, res_max_sweeps - done);
      if ((rc = sweeps(b, v, false, k))) return rc;
      done += k;
    }
    nsw = done;
    return NPHYS_OK;
  }

  // The network's impulses for every row record (features already computed) as the warm start.
  int predict(SolverBufs& v, int C) {
    HIPCK(ml_y.ensure(size_t(C) * kOut * sizeof(float)));
    if (counters_enabled) {
      for (auto& e : ml_ev)
        if (!e) HIPCK(hipEventCreate(&e));
      HIPCK(hipEventRecord(ml_ev[0], stream));
    }
    mlp_infer(MlpDev{ml_img.as<uint16_t>(), ml_params.as<float>()}, ml_X.as<float>(), C, ml_y.as<float>(), stream);
    if (counters_enabled) {
      HIPCK(hipEventRecord(ml_ev[1], stream));
      ml_ev_pending = true;
      ml_rows_pending = C;
    }
    launch_apply_prediction(v, C, ml_y.as<float>(), ml_ls.as<float>(), stream);
    return NPHYS_OK;
  }
  hipEvent_t ml_ev[2] = {nullptr, nullptr};
  bool ml_ev_pending = false;
  int ml_rows_pending = 0;

  // Activation islands and the solved-manifold list (sleeping worlds): sets cv, M and C to the
  // manifolds with an awake dynamic side; the others' cached impulses are carried over.
  int solve_list(const DevBodies& b, ContactBufs& cc, ContactBufs& pc, int prevM, DevContacts& cv, int& M, int& C) {
    const size_t m = size_t(std::max(cc.M, 1)), nn = size_t(std::max(n, 1));
    HIPCK(act_parent.ensure(nn * 4));
    HIPCK(act_can.ensure(nn * 4));
    HIPCK(act_touch.ensure(nn * 4));
    HIPCK(act_mflag[cur].ensure(m * 4));
    HIPCK(act_pos.ensure(m * 4));
    HIPCK(scan.ensure(scan_tiles(m), stream));
    HIPCK(sl_mbody[cur].ensure(m * sizeof(int2)));
    HIPCK(sl_mfirst[cur].ensure(m * 4));
    HIPCK(sl_mcount[cur].ensure(m * 4));
    ActivationBufs a;
    a.parent = act_parent.as<int>();
    a.can = act_can.as<uint32_t>();
    a.touch = act_touch.as<uint32_t>();
    a.mflag = act_mflag[cur].as<uint32_t>();
    a.pos = act_pos.as<uint32_t>();
    a.scan = &scan;
    a.totals = bp_small.as<uint32_t>() + 48;
    fill_u32(a.totals, 0u, 3, stream);
    const DevContacts full = cc.view();
    const JointBufs jv = joint_view();
    launch_activation(b, full, cc.M, a, nj > 0 ? &jv : nullptr, stream);
    DevContacts out = full;
    out.bfirst = nullptr;  // the solved list has no per-body index
    out.bcount = 0;
    out.mbody = sl_mbody[cur].as<int2>();
    out.mfirst = sl_mfirst[cur].as<int>();
    out.mcount = sl_mcount[cur].as<int>();
    launch_solve_list(full, cc.M, a, out, pc.view(), prevM, stream);
    const int rc = readback({{a.totals, 3, 0}});
    if (rc) return rc;
    M = int(rb_host[0]);
    C = int(rb_host[1]);
    active_bodies = int64_t(rb_host[2]);
    cv = out;
    return NPHYS_OK;
  }

  int solve() {
    ++solve_count;  // counts every solve, as the checker does
    ContactBufs& cc = cb[cur];
    ContactBufs& pc = cb[cur ^ 1];
    const int prevM = have_solved ? pc.M : 0;
    DevBodies b = bodies();
    DevContacts cv = cc.view();
    int M = cc.M, C = cc.C;
    if (sleeping) {
      const int rc = solve_list(b, cc, pc, prevM, cv, M, C);
      if (rc) return rc;
    } else {
      active_bodies = n_dynamic;
    }
    sview[cur] = cv;
    sview_M[cur] = M;
    sview_C[cur] = C;
    sview_compact[cur] = sleeping;
    solved_M = M;
    solved_C = C;
    res_inf = res_rms = 0.0;
    res_pending_blocks = -1;  // of a step that failed after its solve
    ncolours = 0;
    if (M == 0 && nj == 0) {
      last_sweeps = res_target > 0.0 ? 0 : prm.max_velocity_iterations;
      counters.velocity_sweeps += last_sweeps;
      HIPCK(hipEventRecord(ev[EV_ASM], stream));
      HIPCK(hipEventRecord(ev[EV_VEL], stream));
      return NPHYS_OK;
    }
    int rc = ensure_solver(M, C);
    if (rc) return rc;
    SolverBufs v = sv_view();
    // the joints' rows (moreau_jean_solver.rs:211-223); the island joints are those neither broken
    // nor removed with an awake dynamic body, decided on the device
    JointBufs jv = joint_view();
    auto joint_rows = [&] {
      if (nj > 0) launch_joint_assemble(b, sp, jv, stream);
    };
    if (M > 0) {
      if ((rc = colour_and_assemble(b, cv, M, C, sp, v, joint_rows))) return rc;
    } else {
      joint_rows();
    }
    HIPCK(hipEventRecord(ev[EV_ASM], stream));
    kt_used = 0;
    choose_variant(M);
    if (tune_pending) HIPCK(hipEventRecord(tune_ev[0], stream));
    if (cur_variant > 0) {
      const int digits = ncolours * (split_order ? 2 : 1);
      HIPCK(sc_info.ensure(size_t(M) * sizeof(int4)));
      HIPCK(sc_rank.ensure(size_t(M) * sizeof(int2)));
      if (nscenes > 1) {
        for (DBuf* d : {&sc_keys, &sc_slot, &sc_keys_alt, &sc_slot_alt}) HIPCK(d->ensure(size_t(M) * 4));
        HIPCK(sc_start.ensure(size_t(nscenes) * size_t(digits + 1) * 4));
        HIPCK(sv_tmp.ensure(radix_temp_words(M) * 4));
        HIPCK(scan.ensure(radix_scan_tiles(M), stream));
        v.tmp = sv_tmp.as<uint32_t>();
      }
      SceneBlocks sc = sc_view();
      launch_scene_order(b, M, nscenes, scene_bits, digits, v, sc, stream);
    }
    const bool learned = contact_model == NPHYS_CONTACT_MODEL_LEARNED_WARMSTART && C > 0;
    if ((learned || capture) && C > 0) {
      HIPCK(ml_X.ensure(size_t(C) * kFeat * sizeof(float)));
      HIPCK(ml_ls.ensure(size_t(C) * sizeof(float)));
      launch_features(b, cv, sp, M, v, ml_X.as<float>(), ml_ls.as<float>(), stream);
    }
    if (learned && judge && res_target > 0.0) {
      // The plain cache warm start is the judge: both solves run from the same assembled system
      // (the same cached impulses, the prediction added to them for the second) and the
      // prediction is kept only when it reaches the residual target in fewer sweeps.
      HIPCK(jd_lam.ensure(size_t(C) * sizeof(float4)));
      HIPCK(jd_lam0.ensure(size_t(C) * sizeof(float4)));
      HIPCK(jd_dv.ensure(size_t(n) * 2 * sizeof(float4)));
      int n_plain = 0, n_learned = 0;
      launch_lam_copy(v, C, jd_lam0.as<float4>(), true, stream);  // the cache warm start
      // the joints' rows start from their cached impulses in both solves
      const size_t jl = size_t(nj) * 2 * sizeof(float4);
      if (nj > 0) {
        HIPCK(jd_jlam.ensure(2 * jl));
        HIPCK(hipMemcpyAsync(jd_jlam.p, j_lam.p, jl, hipMemcpyDeviceToDevice, stream));
      }
      if ((rc = solve_sweeps(b, cv, v, M, C, n_plain))) return rc;
      const double rinf_p = res_inf, rrms_p = res_rms;
      launch_lam_copy(v, C, jd_lam.as<float4>(), true, stream);
      launch_lam_copy(v, C, jd_lam0.as<float4>(), false, stream);
      if (nj > 0) {
        HIPCK(hipMemcpyAsync(jd_jlam.as<char>() + jl, j_lam.p, jl, hipMemcpyDeviceToDevice, stream));
        HIPCK(hipMemcpyAsync(j_lam.p, jd_jlam.p, jl, hipMemcpyDeviceToDevice, stream));
      }
      // the velocity increment is the last 24 bytes of each 64-byte solver block
      char* dv0 = sol.as<char>() + 10 * sizeof(float);
      const size_t pitch = kSolverBlock * sizeof(float4), dvb = 6 * sizeof(float);
      HIPCK(hipMemcpy2DAsync(jd_dv.p, dvb, dv0, pitch, dvb, size_t(n), hipMemcpyDeviceToDevice, stream));
      HIPCK(hipMemset2DAsync(dv0, pitch, 0, dvb, size_t(n), stream));
      if ((rc = predict(v, C))) return rc;
      if ((rc = solve_sweeps(b, cv, v, M, C, n_learned))) return rc;
      const bool keep = n_learned < n_plain;
      if (!keep) {
        launch_lam_copy(v, C, jd_lam.as<float4>(), false, stream);
        if (nj > 0) HIPCK(hipMemcpyAsync(j_lam.p, jd_jlam.as<char>() + jl, jl, hipMemcpyDeviceToDevice, stream));
        HIPCK(hipMemcpy2DAsync(dv0, pitch, jd_dv.p, dvb, dvb, size_t(n), hipMemcpyDeviceToDevice, stream));
        res_inf = rinf_p;
        res_rms = rrms_p;
      }
      counters.judge_plain_sweeps += n_plain;
      counters.judge_learned_sweeps += n_learned;
      counters.judge_kept += keep ? 1 : 0;
      last_sweeps = n_plain + n_learned;
    } else {
      if (learned && (rc = predict(v, C))) return rc;
      if ((rc = solve_sweeps(b, cv, v, M, C, last_sweeps))) return rc;
    }
    if (capture && C > 0) {
      HIPCK(ml_t.ensure(size_t(C) * kOut * sizeof(float)));
      launch_sample_targets(v, C, ml_ls.as<float>(), ml_t.as<float>(), stream);
      samples = C;
    }
    counters.velocity_sweeps += last_sweeps;
    if (res_target > 0.0) launch_cache_impulses(cv, v, M, stream);  // else with the residual
    if (nj > 0) launch_joint_cache(b, sp, jv, stream);
    HIPCK(hipEventRecord(ev[EV_VEL], stream));
    if (keep_colours && M > 0) {
      std::vector<uint32_t> st(M);
      HIPCK(hipMemcpyAsync(st.data(), sv_state2[cur].p, size_t(M) * 4, hipMemcpyDeviceToHost, stream));
      HIPCK(hipStreamSynchronize(stream));
      last_colours.resize(M);
      for (int m = 0; m < M; ++m) last_colours[m] = int(st[m] & 0xffffu);
    }
    return NPHYS_OK;
  }

  int position_correction(const SimParams& ps, int iterations) {
    const bool joints = nj > 0 && !ccd_sub;
    if (sview_M[cur] == 0 && !joints) return NPHYS_OK;
    DevBodies b = bodies();
    SolverBufs v = sv_view();
    JointBufs jv = joint_view();
    if (cur_variant > 0 && !joints) {
      // scene-blocked, as the sweeps of this solve (worlds without joints)
      SceneBlocks sc = sc_view();
      HIPCK(hipEventRecord(fork_ev, stream));
      HIPCK(hipStreamWaitEvent(stream_large, fork_ev, 0));
      launch_position_blocked(b, ps, v, sc, visit_list(), iterations, cur_variant, stream, stream_large);
      HIPCK(hipEventRecord(join_ev, stream_large));
      HIPCK(hipStreamWaitEvent(stream, join_ev, 0));
      return NPHYS_OK;
    }
    // direct launches, runs of two or more consecutive small classes in one workgroup (as the
    // sweeps); the joints' constraints first in every iteration (nonlinear_sor_prox.rs:33-38)
    const int ncol = sview_M[cur] > 0 ? ncolours : 0;
    for (int it = 0; it < iterations; ++it) {
      if (joints) launch_joint_position(b, ps, jv, stream);
      for (int k = 0; k < ncol;) {
        const ClassRun run = small_run(k, ncol);
        if (run.n >= 2) {
          launch_position_run(b, ps, v, run, stream);
          k += run.n;
          continue;
        }
        launch_position_colour(b, ps, h_span[size_t(k)], v, stream);
        ++k;
      }
    }
    return NPHYS_OK;
  }


  // ------------------------------------------------------------------ CCD
  int ensure_ccd() {
    if (n >= kSlotStatic) return set_err(NPHYS_ERR_CAPACITY, "CCD supports fewer than 2^30 bodies");
    const size_t nn = size_t(std::max(n, 1)), P = size_t(std::max(npairs, 1));
    for (DBuf* b : {&ccd_time, &ccd_frozen, &ccd_in, &ccd_new, &ccd_prep, &ccd_prepared, &ccd_deg, &ccd_off, &ccd_fill, &ccd_bodies})
      HIPCK(b->ensure(nn * 4));
    HIPCK(ccd_adj.ensure(2 * P * 4));
    for (DBuf* b : {&ccd_slot, &ccd_stage, &ccd_eval, &ccd_kept, &ccd_cand, &ccd_cpos, &ccd_lpair})
      HIPCK(b->ensure(P * 4));
    HIPCK(ccd_list.ensure(P * sizeof(int2)));
    HIPCK(ccd_sbodies.ensure(P * sizeof(int4)));
    HIPCK(ccd_queue.ensure(P * 8));
    HIPCK(ccd_seen.ensure(2 * P * 8));
    HIPCK(ccd_seen_at.ensure(2 * P * 4));
    HIPCK(ccd_group.ensure(kCcdGroups * 8));
    // the impact list takes 3P + 4096 confirmed impacts (a full list is an error, never a silent loss)
    HIPCK(ccd_imp.ensure((3 * P + 4096) * 8));
    ccd_cap = int(std::min<size_t>(ccd_imp.bytes / 8, size_t(INT_MAX)));
    HIPCK(ccd_ctl.ensure(kCcdWords * 4));
    HIPCK(scan.ensure(std::max(scan_tiles(P), scan_tiles(nn)), stream));
    return NPHYS_OK;
  }

  CcdBufs ccd_view() {
    CcdBufs c;
    c.body_time = ccd_time.as<float>();
    c.frozen = ccd_frozen.as<float>();
    c.slot_pair = ccd_slot.as<int>();
    c.slot_bodies = ccd_sbodies.as<int4>();
    c.key = ccd_queue.as<unsigned long long>();
    c.seen_key = ccd_seen.as<unsigned long long>();
    c.seen_at = ccd_seen_at.as<float>();
    c.group = ccd_group.as<unsigned long long>();
    c.stage = ccd_stage.as<int>();
    c.bodies = ccd_bodies.as<int>();
    c.impacts = ccd_imp.as<unsigned long long>();
    c.ctl = ccd_ctl.as<uint32_t>();
    c.cap = ccd_cap;
    c.in_t = ccd_in.as<uint32_t>();
    c.new_t = ccd_new.as<uint32_t>();
    c.prep = ccd_prep.as<uint32_t>();
    c.prepared = ccd_prepared.as<uint32_t>();
    c.evaluated = ccd_eval.as<uint32_t>();
    c.kept = ccd_kept.as<uint32_t>();
    c.cand = ccd_cand.as<uint32_t>();
    c.cpos = ccd_cpos.as<uint32_t>();
    c.list = ccd_list.as<int2>();
    c.list_pair = ccd_lpair.as<int>();
    c.scan = &scan;
    c.deg = ccd_deg.as<uint32_t>();
    c.off = ccd_off.as<uint32_t>();
    c.fill = ccd_fill.as<uint32_t>();
    c.adj = ccd_adj.as<int>();
    return c;
  }

  // detect() within a step, with its counters.
  int detect_counting(int passes, bool narrow, hipEvent_t bp_done = nullptr, hipEvent_t np_done = nullptr) {
    int64_t changed = 0;
    const bool stale = pairs_dirty;
    const int rc = detect(passes, narrow, &changed, bp_done, np_done);
    if (rc) return rc;
    counters.loose_changes += changed;
    if (changed || stale) ++counters.pair_rebuilds;
    return NPHYS_OK;
  }

  // The CCD phase's sync and broad phase with swept AABBs (position0 -> position).
  int ccd_broad_phase() {
    const int rc = detect_counting(LOOSE_SWEPT, false);
    return rc ? rc : ensure_ccd();
  }

  // predict_next_impacts up to end_time: sets *kind (PREDICT_*), the impact count, the last
  // impact time and min_overstep.
  int ccd_predict(float end_time, float dt0, int* kind) {
    CcdBufs c = ccd_view();
    const DevBodies b = bodies();
    const float target = sp.allowed_linear_error;
    const int on_pen = prm.ccd_on_penetration_enabled;
    (void)hipGetLastError();  // an earlier call's
    launch_ccd_first(b, pairs.as<int2>(), npairs, c, end_time, dt0, target, on_pen, stream);
    // The first batch is one round, which ends it where there are no impacts or few. Every round but the last
    // freezes a body at least, so n + 1 of them end it; a launch that was refused would leave the queue as it is.
    int64_t done = 0;
    for (int rounds = 1;; rounds = 4) {
      for (int k = 0; k < rounds; ++k) launch_ccd_events(b, c, end_time, dt0, target, on_pen, stream);
      HIPCK(hipGetLastError());
      const int rc = readback({{c.ctl, kCcdWords, 0}});
      if (rc) return rc;
      if (rb_host[kCcdOverflow]) return set_err(NPHYS_ERR_CAPACITY, "CCD impact queue overflow");
      if (rb_host[kCcdState] == kQueueDone) break;
      if ((done += rounds) > n) return set_err(NPHYS_ERR_STATE, "CCD impact queue did not end");
    }
    *kind = int(rb_host[kCcdKind]);
    ccd_nimp = *kind == PREDICT_IMPACTS ? int(rb_host[kCcdImpacts]) : 0;
    uint32_t u = rb_host[kCcdLastToi];
    std::memcpy(&ccd_last_toi, &u, 4);
    u = rb_host[kCcdMinOver];
    std::memcpy(&ccd_min_over, &u, 4);
    return NPHYS_OK;
  }

  // One substep (mechanical_world.rs:630-935): the island moved to the last impact time, its
  // manifolds at the moved poses, then MoreauJeanSolver::step_ccd over dt0 - last_toi: assembly
  // without warm start (coefficient 0), max_ccd_position_iterations position iterations, the
  // impacting bodies' advancement validated, the velocity sweeps, integration of the island.
  int ccd_substep(float dt0) {
    int rc;
    ++counters.ccd_substeps;
    counters.ccd_impacts += ccd_nimp;
    const float last_toi = ccd_last_toi;
    const float dt_sub = dt0 - last_toi;
    const DevBodies b = bodies();
    CcdBufs c = ccd_view();
    launch_ccd_island(n, std::max(npairs, 1), c, stream);
    launch_ccd_seed(b, pairs.as<int2>(), c, ccd_nimp, stream);
    for (;;) {  // island rounds
      launch_ccd_touch(b, pairs.as<int2>(), npairs, c, stream);
      launch_ccd_prepare(b, c, dt_sub, last_toi, stream);
      launch_ccd_compact(pairs.as<int2>(), npairs, c.cand, c, stream);
      if ((rc = readback({{c.ctl + kCcdList, 1, 0}}))) return rc;
      const int nl = int(rb_host[0]);
      if (nl == 0) break;
      if ((rc = narrow_phase_of(c.list, nl, c.ctl + kCcdList, ccd_cb, false))) return rc;
      launch_ccd_grow(b, c, nl, np_count.as<uint32_t>(), stream);
      launch_ccd_merge(n, c, stream);
    }
    // the island's manifolds, in pair order, into cb[cur] (the final narrow phase rewrites it)
    launch_ccd_compact(pairs.as<int2>(), npairs, c.kept, c, stream);
    if ((rc = readback({{c.ctl + kCcdList, 1, 0}}))) return rc;
    const int nk = int(rb_host[0]);
    ContactBufs& cc = cb[cur];
    if ((rc = narrow_phase_of(c.list, nk, c.ctl + kCcdList, cc))) return rc;
    const int M = cc.M, C = cc.C;
    SimParams ss = sp;
    ss.dt = dt_sub;
    ss.inv_dt = dt_sub == 0.0f ? 0.0f : 1.0f / dt_sub;
    ss.warmstart_coeff = 0.0f;
    ss.gx = ss.gy = ss.gz = 0.0f;
    ss.dyn_dt = dt_sub;
    const DevContacts cv = cc.view();
    ++solve_count;
    ccd_sub = true;
    const int saved_variant = cur_variant;
    cur_variant = 0;
    SolverBufs v{};
    if (M > 0) {
      if ((rc = ensure_solver(M, C))) return rc;
      v = sv_view();
      if ((rc = colour_and_assemble(b, cv, M, C, ss, v, [] {}))) return rc;
      sview[cur] = cv;
      sview_M[cur] = M;
      sview_C[cur] = C;
      if ((rc = position_correction(ss, prm.max_ccd_position_iterations))) return rc;
    }
    launch_ccd_validate(b, pairs.as<int2>(), c, ccd_nimp, stream);
    if (M > 0 && (rc = sweeps(b, v, true, prm.max_velocity_iterations))) return rc;
    launch_integrate(b, ss, stream, c.prepared);
    ccd_sub = false;
    cur_variant = saved_variant;
    // every moved body's dynamics are updated with the substep's time step after it (:915-923)
    dyn_dt_next = dt_sub;
    return NPHYS_OK;
  }

  // MechanicalWorld::solve_ccd (mechanical_world.rs:559-943).
  int solve_ccd() {
    int rc;
    const float dt0 = sp.dt;
    if (dt0 == 0.0f || prm.max_ccd_substeps == 0) return NPHYS_OK;
    const float sub_len = dt0 / float(prm.max_ccd_substeps);
    if ((rc = ensure_ccd())) return rc;
    fill_u32(ccd_time.as<uint32_t>(), 0u, size_t(n), stream);
    float end_time = 0.0f;
    bool last_iter = false;
    for (;;) {
      if (end_time < dt0) end_time = fminf_(end_time + sub_len, dt0);
      else last_iter = true;
      if ((rc = ccd_broad_phase())) return rc;
      int kind = PREDICT_NONE;
      if ((rc = ccd_predict(end_time, dt0, &kind))) return rc;
      if (kind == PREDICT_AFTER_END) {
        end_time = std::floor(ccd_min_over / sub_len) * sub_len;
        end_time = fminf_(end_time + sub_len, dt0);
        if ((rc = ccd_predict(end_time, dt0, &kind))) return rc;
        if (kind != PREDICT_IMPACTS) return set_err(NPHYS_ERR_STATE, "CCD: no impact in the window of the earliest one");
      }
      if (!last_iter && ccd_nimp > 0) {
        if ((rc = ccd_substep(dt0))) return rc;
        continue;
      }
      CcdBufs c = ccd_view();
      launch_ccd_clamp(bodies(), c, stream);  // the last prediction's frozen bodies
      return NPHYS_OK;
    }
  }

  // ------------------------------------------------------------------ step
  int step_once() {
    int rc;
    HIPCK(hipEventRecord(ev[EV_START], stream));
    // bodies moved from the host are updated at their new state with this step's dt; the others
    // keep the time step of their last update (a CCD substep's after one)
    SimParams spp = sp;
    spp.dyn_dt = moved ? sp.dt : dyn_dt_next;
    dyn_dt_next = sp.dt;
    if (moved || recollide) {
      if ((rc = collide_now())) return rc;
      moved = false;
      recollide = false;
    }
    HIPCK(hipEventRecord(ev[EV_PRE_CD], stream));
    if (wake_pending) {
      launch_wake(bodies(), stream);
      wake_pending = false;
    }
    launch_prestep(bodies(), spp, stream);
    if ((rc = solve())) return rc;
    launch_integrate(bodies(), sp, stream);
    HIPCK(hipEventRecord(ev[EV_INT], stream));
    if ((rc = position_correction(sp, prm.max_position_iterations))) return rc;
    HIPCK(hipEventRecord(ev[EV_POS], stream));
    if (tune_pending) HIPCK(hipEventRecord(tune_ev[1], stream));  // the variant's sweeps and position passes
    // this step's manifolds and impulses become the warm-start cache
    cur ^= 1;
    have_solved = true;
    if (any_ccd) {
      // the CCD phase (its swept syncs and broad phases, impacts and substeps), then the final sync
      if ((rc = solve_ccd())) return rc;
      HIPCK(hipEventRecord(ev[EV_CCD], stream));
      rc = detect_counting(LOOSE_FINAL, true, ev[EV_BP], ev[EV_NP]);
    } else {
      // the CCD phase's swept sync, which solve_ccd's loop returns before when dt or max_ccd_substeps
      // is zero (mechanical_world.rs:578-581), then the final one
      HIPCK(hipEventRecord(ev[EV_CCD], stream));
      const bool swept = sp.dt != 0.0f && prm.max_ccd_substeps != 0;
      rc = detect_counting(LOOSE_FINAL | (swept ? LOOSE_SWEPT : 0), true, ev[EV_BP], ev[EV_NP]);
    }
    // the detection's readback completes the step: every earlier event and copy is done after it
    if (rc) return rc;
    finish_residual();
    auto el = [&](int a, int c) {
      float ms = 0.0f;
      (void)hipEventElapsedTime(&ms, ev[a], ev[c]);
      return double(ms) * 1e-3;
    };
    counters.step += el(EV_START, EV_NP);
    counters.collision_detection += el(EV_START, EV_PRE_CD) + el(EV_CCD, EV_NP);
    counters.broad_phase += el(EV_CCD, EV_BP);
    counters.ccd_time += el(EV_POS, EV_CCD);
    counters.narrow_phase += el(EV_BP, EV_NP);
    counters.assembly += el(EV_PRE_CD, EV_ASM);
    counters.velocity_resolution += el(EV_ASM, EV_VEL);
    counters.velocity_update += el(EV_VEL, EV_INT);
    counters.position_resolution += el(EV_INT, EV_POS);
    counters.nsteps += 1;
    counters.npairs = npairs;
    counters.ncontacts = solved_C;
    counters.nmanifolds = solved_M;
    counters.active_bodies = active_bodies;
    counters.nconstraints = int64_t(3) * solved_C;
    counters.ncolours = ncolours;
    counters.colour_rounds += colour_rounds;
    tune_record();
    counters.sweep_variant = cur_variant;
    for (int k = 0; k < kt_used; k += 2) {
      float ms = 0.0f;
      (void)hipEventElapsedTime(&ms, kt_ev[k], kt_ev[k + 1]);
      counters.sweep_kernel_time += double(ms) * 1e-3;
      counters.sweep_kernel_launches += 1;
    }
    kt_used = 0;
    if (ml_ev_pending) {  // the step's final synchronisation has passed the inference
      float ms = 0.0f;
      if (hipEventElapsedTime(&ms, ml_ev[0], ml_ev[1]) == hipSuccess) {
        counters.warmstart_inference_time += double(ms) * 1e-3;
        counters.warmstart_inference_rows += ml_rows_pending;
      }
      ml_ev_pending = false;
    }
    prm.t += prm.dt;
    // clear_forces (mechanical_world.rs:365): the next accumulation starts from zero
    if (forces_pending) {
      fill_u32(f_lin.as<uint32_t>(), 0u, size_t(n) * 4, stream);
      fill_u32(f_ang.as<uint32_t>(), 0u, size_t(n) * 4, stream);
      forces_pending = false;
    }
    rot_dyn_saved = false;
    return NPHYS_OK;
  }

  // Body::apply_force / apply_force_at_point for `count` entries: grouped by body on the host (a
  // stable sort keeps each body's entries in the caller's order), one thread per body.
  int apply_force(int32_t count, const int32_t* bodies_, const float* forces, const float* points, int32_t type,
                  int32_t wake) {
    if (count < 0 || type < 0 || type > 3) return set_err(NPHYS_ERR_INVALID, "bad force arguments");
    if (count == 0) return NPHYS_OK;
    if (!bodies_ || !forces) return set_err(NPHYS_ERR_INVALID, "null force arrays");
    for (int k = 0; k < count; ++k)
      if (bodies_[k] < 0 || bodies_[k] >= n) return set_err(NPHYS_ERR_INVALID, "bad body handle");
    std::vector<int> order(static_cast<size_t>(count));
    for (int k = 0; k < count; ++k) order[size_t(k)] = k;
    std::stable_sort(order.begin(), order.end(), [&](int a, int c) { return bodies_[a] < bodies_[c]; });
    std::vector<int> ub, off;
    for (int k = 0; k < count; ++k) {
      const int bd = bodies_[order[size_t(k)]];
      if (ub.empty() || ub.back() != bd) {
        ub.push_back(bd);
        off.push_back(k);
      }
    }
    off.push_back(count);
    const int nu = int(ub.size());
    const int fw = points ? 3 : 6;
    const size_t words = size_t(nu) + size_t(nu + 1) + size_t(count) + size_t(count) * fw + (points ? size_t(count) * 3 : 0);
    HIPCK(af_tmp.ensure(words * 4));
    char* base = af_tmp.as<char>();
    int* d_ub = reinterpret_cast<int*>(base);
    int* d_off = d_ub + nu;
    int* d_order = d_off + nu + 1;
    float* d_f = reinterpret_cast<float*>(d_order + count);
    float* d_p = points ? d_f + size_t(count) * fw : nullptr;
    HIPCK(hipMemcpyAsync(d_ub, ub.data(), size_t(nu) * 4, hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(d_off, off.data(), size_t(nu + 1) * 4, hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(d_order, order.data(), size_t(count) * 4, hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(d_f, forces, size_t(count) * fw * 4, hipMemcpyHostToDevice, stream));
    if (points) HIPCK(hipMemcpyAsync(d_p, points, size_t(count) * 12, hipMemcpyHostToDevice, stream));
    if (type == NPHYS_FORCE || type == NPHYS_ACCELERATION_CHANGE) forces_pending = true;
    SimParams spf = sp;
    spf.dyn_dt = dyn_dt_next;  // the time step of the augmented mass the forces act through
    launch_apply_force(bodies(), spf, nu, d_ub, d_off, d_order, d_f, d_p, type, wake, rot_dyn_saved ? rot_dyn.as<float4>() : nullptr,
                       stream);
    HIPCK(hipStreamSynchronize(stream));  // the staging buffer is reused by the next call
    return NPHYS_OK;
  }

  // MaterialsCoefficientsTable::set_friction_coefficient / set_restitution_coefficient.
  int set_material_coefficient(int32_t which, int32_t id1, int32_t id2, float coeff) {
    if ((which != 0 && which != 1) || id1 < 0 || id2 < 0) return set_err(NPHYS_ERR_INVALID, "bad material pair");
    const unsigned long long lo = unsigned(std::min(id1, id2)), hi = unsigned(std::max(id1, id2));
    const unsigned long long key = (lo << 32) | hi;
    auto& t = mt_host[which];
    auto it = std::lower_bound(t.begin(), t.end(), std::make_pair(key, -std::numeric_limits<float>::infinity()),
                               [](const std::pair<unsigned long long, float>& a,
                                  const std::pair<unsigned long long, float>& c) { return a.first < c.first; });
    if (it != t.end() && it->first == key) {
      it->second = coeff;
    } else {
      if (t.size() >= NPHYS_MAX_MATERIAL_PAIRS) return set_err(NPHYS_ERR_CAPACITY, "material table full");
      t.insert(it, std::make_pair(key, coeff));
    }
    std::vector<unsigned long long> keys(t.size());
    std::vector<float> vals(t.size());
    for (size_t i = 0; i < t.size(); ++i) {
      keys[i] = t[i].first;
      vals[i] = t[i].second;
    }
    HIPCK(hipStreamSynchronize(stream));  // the previous table may be read by enqueued work
    HIPCK(mt_key[which].ensure(keys.size() * 8));
    HIPCK(mt_val[which].ensure(vals.size() * 4));
    HIPCK(hipMemcpyAsync(mt_key[which].p, keys.data(), keys.size() * 8, hipMemcpyHostToDevice, stream));
    HIPCK(hipMemcpyAsync(mt_val[which].p, vals.data(), vals.size() * 4, hipMemcpyHostToDevice, stream));
    HIPCK(hipStreamSynchronize(stream));
    return NPHYS_OK;
  }
};

}  // namespace nph

using nph::World;
using nph::set_err;

struct nphys_world {
  World w;
};

extern "C" {

void nphys_params_default(nphys_params* out) {
  if (!out) return;
  std::memset(out, 0, sizeof(*out));
  out->t = 0.0;
  out->dt = 1.0 / 60.0;
  out->erp = 0.2;
  out->warmstart_coeff = 1.0;
  out->restitution_velocity_threshold = 1.0;
  out->allowed_linear_error = 0.001;
  out->allowed_angular_error = 0.001;
  out->max_linear_correction = 0.2;
  out->max_angular_correction = 0.2;
  out->max_stabilization_multiplier = 0.2;
  out->max_velocity_iterations = 8;
  out->max_position_iterations = 3;
  out->max_ccd_position_iterations = 10;
  out->max_ccd_substeps = 1;
  out->gravity[0] = 0.0;
  out->gravity[1] = -9.81;
  out->gravity[2] = 0.0;
}

static int check_params(const nphys_params* p) {
  if (!p) return set_err(NPHYS_ERR_INVALID, "null params");
  if (!(p->dt >= 0.0)) return set_err(NPHYS_ERR_INVALID, "dt must be non-negative");
  if (p->max_velocity_iterations < 0 || p->max_position_iterations < 0)
    return set_err(NPHYS_ERR_INVALID, "negative iteration count");
  return NPHYS_OK;
}

int nphys_world_create(const nphys_params* params, nphys_world** out) {
  if (!out) return set_err(NPHYS_ERR_INVALID, "null out");
  *out = nullptr;
  int rc = check_params(params);
  if (rc) return rc;
  nphys_world* w = new nphys_world();
  rc = w->w.init(*params);
  if (rc) {
    delete w;
    return rc;
  }
  *out = w;
  return NPHYS_OK;
}

int nphys_world_destroy(nphys_world* w) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  if (w->w.stream) (void)hipStreamSynchronize(w->w.stream);
  delete w;
  return NPHYS_OK;
}

int nphys_set_params(nphys_world* w, const nphys_params* params) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  const int rc = check_params(params);
  if (rc) return rc;
  w->w.set_params(*params);
  return NPHYS_OK;
}

int nphys_get_params(const nphys_world* w, nphys_params* out) {
  if (!w || !out) return set_err(NPHYS_ERR_INVALID, "null argument");
  *out = w->w.prm;
  return NPHYS_OK;
}

int nphys_add_bodies(nphys_world* w, const nphys_body_desc* desc, int32_t* first_handle) {
  if (!w || !desc) return set_err(NPHYS_ERR_INVALID, "null argument");
  return w->w.add_bodies(*desc, first_handle);
}

int nphys_add_joints(nphys_world* w, const nphys_joint_desc* desc, int32_t* first_handle) {
  if (!w || !desc) return set_err(NPHYS_ERR_INVALID, "null argument");
  return w->w.add_joints(*desc, first_handle);
}

int nphys_remove_joint(nphys_world* w, int32_t joint) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  return w->w.remove_joint(joint);
}

int nphys_num_joints(const nphys_world* w, int32_t* n) {
  if (!w || !n) return set_err(NPHYS_ERR_INVALID, "null argument");
  *n = w->w.nj;
  return NPHYS_OK;
}

int nphys_read_joints(nphys_world* w, float* lin_impulses, float* ang_impulses, int32_t* broken, int64_t cap) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  return w->w.read_joints(lin_impulses, ang_impulses, broken, cap);
}

int nphys_num_bodies(const nphys_world* w, int32_t* n) {
  if (!w || !n) return set_err(NPHYS_ERR_INVALID, "null argument");
  *n = w->w.n;
  return NPHYS_OK;
}

int nphys_set_state(nphys_world* w, const float* pos, const float* rot, const float* linvel,
                    const float* angvel) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  return w->w.set_state(pos, rot, linvel, angvel);
}

int nphys_set_collision_groups(nphys_world* w, int32_t count, const int32_t* bodies, const uint32_t* groups) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  return w->w.set_collision_groups(count, bodies, groups);
}

int nphys_get_state(nphys_world* w, float* pos, float* rot, float* linvel, float* angvel) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  return w->w.get_state(pos, rot, linvel, angvel);
}

int nphys_apply_force(nphys_world* w, int32_t count, const int32_t* bodies, const float* forces, int32_t type,
                      int32_t auto_wake_up) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  return w->w.apply_force(count, bodies, forces, nullptr, type, auto_wake_up);
}

int nphys_apply_force_at_point(nphys_world* w, int32_t count, const int32_t* bodies, const float* forces,
                               const float* points, int32_t type, int32_t auto_wake_up) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  if (count > 0 && !points) return set_err(NPHYS_ERR_INVALID, "null points");
  return w->w.apply_force(count, bodies, forces, points, type, auto_wake_up);
}

int nphys_set_material_coefficient(nphys_world* w, int32_t which, int32_t id1, int32_t id2, float coeff) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  return w->w.set_material_coefficient(which, id1, id2, coeff);
}

int nphys_step(nphys_world* w, int32_t nsteps) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  if (nsteps < 0) return set_err(NPHYS_ERR_INVALID, "negative step count");
  if (w->w.any_ccd && (w->w.sleeping || w->w.nscenes > 1))
    return set_err(NPHYS_ERR_INVALID, "CCD needs one scene and no sleep thresholds");
  for (int i = 0; i < nsteps; ++i) {
    const int rc = w->w.step_once();
    if (rc) return rc;
  }
  return NPHYS_OK;
}

int nphys_collide(nphys_world* w) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  const int rc = w->w.collide_now();
  if (rc) return rc;
  w->w.moved = false;
  w->w.recollide = false;
  if (hipStreamSynchronize(w->w.stream) != hipSuccess) return set_err(NPHYS_ERR_HIP, "sync failed");
  return NPHYS_OK;
}

int nphys_contact_model_set(nphys_world* w, int32_t model) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  if (model != NPHYS_CONTACT_MODEL_SIGNORINI_COULOMB_PYRAMID && model != NPHYS_CONTACT_MODEL_LEARNED_WARMSTART)
    return set_err(NPHYS_ERR_INVALID, "unknown contact model");
  if (model == NPHYS_CONTACT_MODEL_LEARNED_WARMSTART && !w->w.ml_loaded)
    return set_err(NPHYS_ERR_STATE, "the learned warm start needs a network (nphys_warmstart_load)");
  w->w.contact_model = model;
  return NPHYS_OK;
}

int nphys_warmstart_load(nphys_world* w, const float* params, int64_t n) {
  if (!w || !params) return set_err(NPHYS_ERR_INVALID, "null argument");
  if (n != nph::kNumParams) return set_err(NPHYS_ERR_INVALID, "parameter count mismatch");
  for (int i = 0; i < nph::kFeat; ++i)
    if (!(params[nph::kOffXScale + i] > 0.0f)) return set_err(NPHYS_ERR_INVALID, "feature scales must be > 0");
  for (int i = 0; i < nph::kOut; ++i)
    if (!(params[nph::kOffYScale + i] > 0.0f)) return set_err(NPHYS_ERR_INVALID, "output scales must be > 0");
  World& W = w->w;
  HIPCK(W.ml_params.ensure(size_t(nph::kNumParams) * 4));
  HIPCK(W.ml_img.ensure(size_t(nph::kImgElems) * 2));
  HIPCK(hipMemcpyAsync(W.ml_params.p, params, size_t(nph::kNumParams) * 4, hipMemcpyHostToDevice, W.stream));
  nph::mlp_pack_images(W.ml_params.as<float>(), W.ml_img.as<uint16_t>(), W.stream);
  HIPCK(hipStreamSynchronize(W.stream));
  W.ml_loaded = true;
  return NPHYS_OK;
}

int nphys_capture_samples(nphys_world* w, int32_t on) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  w->w.capture = on != 0;
  w->w.samples = 0;
  return NPHYS_OK;
}

int nphys_read_samples(nphys_world* w, float* features, float* targets, int64_t cap, int64_t* n) {
  if (!w || !n) return set_err(NPHYS_ERR_INVALID, "null argument");
  World& W = w->w;
  *n = W.samples;
  if (!features && !targets) return NPHYS_OK;
  if (cap < W.samples) return set_err(NPHYS_ERR_CAPACITY, "sample buffers too small");
  if (W.samples == 0) return NPHYS_OK;
  if (features)
    HIPCK(hipMemcpyAsync(features, W.ml_X.p, size_t(W.samples) * nph::kFeat * 4, hipMemcpyDeviceToHost, W.stream));
  if (targets)
    HIPCK(hipMemcpyAsync(targets, W.ml_t.p, size_t(W.samples) * nph::kOut * 4, hipMemcpyDeviceToHost, W.stream));
  HIPCK(hipStreamSynchronize(W.stream));
  return NPHYS_OK;
}

int nphys_set_sweep_variant(nphys_world* w, int32_t variant) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  if (variant != -1 && variant != 0 && variant != 256 && variant != 512 && variant != 1024)
    return set_err(NPHYS_ERR_INVALID, "variant must be -1 (autotune), 0, 256, 512 or 1024");
  w->w.variant_request = variant;
  w->w.tune_cands.clear();
  w->w.tuned = false;
  return NPHYS_OK;
}

// For the tests, and so not in the header: a smaller limit than kMostPairs for this world (at least 1: no
// launch of the narrow phase is for fewer pairs).
int nphys_test_most_pairs(nphys_world* w, int32_t pairs) {
  if (!w || pairs < 1 || pairs > nph::World::kMostPairs) return set_err(NPHYS_ERR_INVALID, "bad argument");
  w->w.most_pairs = pairs;
  return NPHYS_OK;
}

int nphys_set_incremental_pairs(nphys_world* w, int32_t on) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  w->w.incremental_bp = on != 0;
  return NPHYS_OK;
}

int nphys_set_warmstart_judge(nphys_world* w, int32_t on) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  w->w.judge = on != 0;
  return NPHYS_OK;
}

int nphys_num_pairs(nphys_world* w, int64_t* n) {
  if (!w || !n) return set_err(NPHYS_ERR_INVALID, "null argument");
  *n = w->w.npairs;
  return NPHYS_OK;
}

int nphys_read_pairs(nphys_world* w, int32_t* pairs, int64_t cap) {
  if (!w || (!pairs && w->w.npairs)) return set_err(NPHYS_ERR_INVALID, "null argument");
  if (cap < w->w.npairs) return set_err(NPHYS_ERR_CAPACITY, "pair buffer too small");
  if (w->w.npairs == 0) return NPHYS_OK;
  return w->w.pairs_out(pairs);
}

int nphys_num_contacts(nphys_world* w, int64_t* n) {
  if (!w || !n) return set_err(NPHYS_ERR_INVALID, "null argument");
  *n = w->w.cb[w->w.cur].C;
  return NPHYS_OK;
}

int nphys_read_contacts(nphys_world* w, int32_t* bodies, uint32_t* feature, float* world1,
                        float* world2, float* normal, float* depth, int64_t cap) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  nph::ContactBufs& c = w->w.cb[w->w.cur];
  if (cap < c.C) return set_err(NPHYS_ERR_CAPACITY, "contact buffer too small");
  if (c.C == 0) return NPHYS_OK;
  return w->w.contacts_out(c, nph::ContactRows{{reinterpret_cast<float*>(bodies), reinterpret_cast<float*>(feature),
                                                world1, world2, normal, depth}});
}

int nphys_num_manifolds(nphys_world* w, int64_t* n) {
  if (!w || !n) return set_err(NPHYS_ERR_INVALID, "null argument");
  *n = w->w.cb[w->w.cur].M;
  return NPHYS_OK;
}

int nphys_read_manifolds(nphys_world* w, int32_t* bodies, int32_t* first, int32_t* count, int64_t cap) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  nph::ContactBufs& c = w->w.cb[w->w.cur];
  if (cap < c.M) return set_err(NPHYS_ERR_CAPACITY, "manifold buffer too small");
  if (c.M == 0) return NPHYS_OK;
  std::vector<int2> mb(static_cast<size_t>(c.M));
  std::vector<int> mc(static_cast<size_t>(c.M));
  HIPCK(hipMemcpyAsync(mb.data(), c.mbody.p, mb.size() * sizeof(int2), hipMemcpyDeviceToHost, w->w.stream));
  HIPCK(hipMemcpyAsync(mc.data(), c.mcount.p, mc.size() * 4, hipMemcpyDeviceToHost, w->w.stream));
  HIPCK(hipStreamSynchronize(w->w.stream));
  int32_t acc = 0;
  for (size_t m = 0; m < mb.size(); ++m) {
    if (bodies) {
      bodies[2 * m] = mb[m].x;
      bodies[2 * m + 1] = mb[m].y;
    }
    if (first) first[m] = acc;
    if (count) count[m] = mc[m];
    acc += mc[m];
  }
  return NPHYS_OK;
}

int nphys_num_solved_contacts(nphys_world* w, int64_t* n) {
  if (!w || !n) return set_err(NPHYS_ERR_INVALID, "null argument");
  *n = w->w.have_solved ? w->w.sview_C[w->w.cur ^ 1] : 0;
  return NPHYS_OK;
}

int nphys_read_impulses(nphys_world* w, uint64_t* keys, float* impulses, int64_t cap) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  if (!w->w.have_solved) return NPHYS_OK;
  const int par = w->w.cur ^ 1;
  nph::ContactBufs& c = w->w.cb[par];
  if (cap < w->w.sview_C[par]) return set_err(NPHYS_ERR_CAPACITY, "impulse buffer too small");
  if (w->w.sview_C[par] == 0) return NPHYS_OK;
  std::vector<int2> mb;
  std::vector<int> mc;
  std::vector<float4> rec, imp;
  int rc = w->w.gather_contacts(c, mb, mc, rec, &imp);
  if (rc) return rc;
  // sleeping worlds: only the manifolds handed to the solver
  std::vector<uint32_t> solved;
  if (w->w.sview_compact[par]) {
    solved.resize(mb.size());
    if (!solved.empty()) {
      HIPCK(hipMemcpyAsync(solved.data(), w->w.act_mflag[par].p, solved.size() * 4, hipMemcpyDeviceToHost,
                           w->w.stream));
      HIPCK(hipStreamSynchronize(w->w.stream));
    }
  }
  long i = 0, j = 0;
  for (size_t m = 0; m < mb.size(); ++m)
    for (int k = 0; k < mc[m]; ++k, ++j) {
      if (!solved.empty() && !solved[m]) continue;
      const uint32_t f = nph::bits_of(rec[size_t(j) * nph::kContactFields + 1].w);
      if (keys)
        keys[i] = (uint64_t(uint32_t(mb[m].x)) << 40) | (uint64_t(uint32_t(mb[m].y)) << 16) | uint64_t(f & 0xffffu);
      if (impulses) {
        impulses[3 * i] = imp[size_t(j)].x;
        impulses[3 * i + 1] = imp[size_t(j)].y;
        impulses[3 * i + 2] = imp[size_t(j)].z;
      }
      ++i;
    }
  return NPHYS_OK;
}

int nphys_residual(nphys_world* w, double* r_inf, double* r_rms) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  if (r_inf) *r_inf = w->w.res_inf;
  if (r_rms) *r_rms = w->w.res_rms;
  return NPHYS_OK;
}

int nphys_read_counters(nphys_world* w, nphys_counters* out) {
  if (!w || !out) return set_err(NPHYS_ERR_INVALID, "null argument");
  *out = w->w.counters;
  return NPHYS_OK;
}

int nphys_reset_counters(nphys_world* w) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  std::memset(&w->w.counters, 0, sizeof(w->w.counters));
  return NPHYS_OK;
}

int nphys_counters_enable(nphys_world* w, int32_t enabled) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  w->w.counters_enabled = enabled != 0;
  return NPHYS_OK;
}

int nphys_set_residual_target(nphys_world* w, double target, int32_t max_sweeps, int32_t check_every,
                              int32_t norm) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  if (!(target >= 0.0) || max_sweeps < 0 || check_every < 1 ||
      (norm != NPHYS_RESIDUAL_MAX && norm != NPHYS_RESIDUAL_RMS))
    return set_err(NPHYS_ERR_INVALID, "target >= 0, max_sweeps >= 0, check_every >= 1, norm MAX or RMS");
  w->w.res_target = target;
  w->w.res_max_sweeps = max_sweeps;
  w->w.res_check_every = check_every;
  w->w.res_norm = norm;
  return NPHYS_OK;
}

int nphys_read_activation(nphys_world* w, float* energy, int64_t cap) {
  if (!w || !energy) return set_err(NPHYS_ERR_INVALID, "null argument");
  return w->w.read_activation(energy, cap);
}

int nphys_read_colours(nphys_world* w, int32_t* colours, int64_t cap, int32_t* ncolours) {
  if (!w) return set_err(NPHYS_ERR_INVALID, "null world");
  w->w.keep_colours = true;
  const int M = int(w->w.last_colours.size());
  if (ncolours) *ncolours = w->w.ncolours;
  if (!colours) return NPHYS_OK;
  if (cap < M) return set_err(NPHYS_ERR_CAPACITY, "colour buffer too small");
  for (int m = 0; m < M; ++m) colours[m] = w->w.last_colours[m];
  return NPHYS_OK;
}

const char* nphys_last_error(void) { return nph::g_err.c_str(); }

}  // extern "C"
