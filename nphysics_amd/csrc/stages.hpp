// nphysics_amd/csrc/stages.hpp -- launch wrappers of the per-stage kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "devworld.hpp"
#include "kernels.hpp"

namespace nph {

// k_bodies.hip
void launch_prestep(const DevBodies& b, const SimParams& p, hipStream_t s);
// only: when given, the bodies with only[i] != 0 (a CCD substep's island)
void launch_integrate(const DevBodies& b, const SimParams& p, hipStream_t s, const uint32_t* only = nullptr);
void launch_clear_dyn_marks(const DevBodies& b, hipStream_t s);
// Packed rows of the bodies' state in pinned host memory as the device addresses it: positions (3
// floats per body), rotations (4), linear and angular velocities (3 each), each 16-byte aligned; null:
// not moved. Velocities are set for dynamic bodies only.
struct StateRows {
  float* row[4];
};
void launch_state_out(const DevBodies& b, const StateRows& o, hipStream_t s);
void launch_state_in(const DevBodies& b, const StateRows& o, hipStream_t s);

void launch_save_rot_dyn(const DevBodies& b, float4* out, hipStream_t s);
void launch_apply_force(const DevBodies& b, const SimParams& p, int nu, const int* ubody, const int* off,
                        const int* order, const float* forces, const float* points, int type, int wake,
                        const float4* rot_dyn, hipStream_t s);

// k_activation.hip ------------------------------------------------------------------------
struct ActivationBufs {
  int* parent;       // [n] union-find parents
  uint32_t* can;     // [n] per island root: every body may sleep
  uint32_t* touch;   // [n] body that could sleep touches one that keeps its island awake
  uint32_t* mflag;   // [M] manifold handed to the solver
  uint32_t* pos;     // [M] its index in the solved list
  ScanState* scan;
  uint32_t* totals;  // [3] solved manifolds, their contacts, awake dynamic bodies (zeroed by the caller)
};
void launch_wake(const DevBodies& b, hipStream_t s);
struct JointBufs;
// j (may be null): joints whose bodies join the islands
void launch_activation(const DevBodies& b, const DevContacts& c, int M, const ActivationBufs& a, const JointBufs* j,
                       hipStream_t s);
void launch_solve_list(const DevContacts& c, int M, const ActivationBufs& a, const DevContacts& out,
                       const DevContacts& prev, int prevM, hipStream_t s);

// k_broadphase.hip ------------------------------------------------------------------------
struct BroadPhaseBufs {
  uint32_t* changed;      // [4] number of loose AABBs replaced (all, of non-dynamic bodies) by the
                          // swept pass and by the other
  uint32_t* bounds;       // [6] ordered-int encoded centroid bounds
  uint32_t* keys;         // [n] Morton codes
  uint32_t* vals;         // [n] the order: body indices
  uint32_t* keys_alt;
  uint32_t* vals_alt;
  float4* leaf_mn;        // [n] loose AABBs in the order, with index and dynamic flag
  float4* leaf_mx;        //     and scene
  float4* box_mn;         // [search_boxes(n)] boxes of 64 of them, then boxes of 64 boxes, with first
  float4* box_mx;         //     and last scene
  int* box_top;           // and the largest index of a partner in them
  int scene_bits;         // Morton keys carry the scene in their top scene_bits bits
  int* cand;              // [n * cap] candidate partners per body
  uint32_t* cand_count;   // [n] partner count (may exceed cap)
  uint32_t* stats;        // [1] largest partner count above the capacity (else 0)
  int2* pairs;            // [pair capacity]
  uint32_t* tmp;          // radix scratch
  ScanState* scan;
  uint32_t* dirty;        // [n] 1 where the loose AABB was replaced since the last pair build
  int* list;              // [n] dirty bodies
  uint32_t* list_count;   // [1]
};

// Loose-AABB passes, as bits: the current pose of the dynamic bodies (1), first the AABB swept from
// pos0/rot0 to pos/rot (2), the static bodies' current pose too (4).
enum : int { LOOSE_FINAL = 1, LOOSE_SWEPT = 2, LOOSE_STATIC = 4 };
void launch_loose_update(const DevBodies& b, int passes, BroadPhaseBufs& bp, hipStream_t s);
// Boxes of n colliders and boxes of those.
inline size_t search_boxes(size_t n) { return (n + 63) / 64 + (n + 4095) / 4096; }
// The order of the colliders (by scene and Morton code), sorted anew.
void launch_order(const DevBodies& b, BroadPhaseBufs& bp, hipStream_t s);
// A pair search: directly, with the end of the last non-dynamic collider, or by boxes over the order;
// the segment capacity, and whether segments may be kept.
// Segments are kept while at most this many of n bodies are dirty: every clean body tests them all,
// which at 1,024 costs as much as a search of its own.
__host__ __device__ inline int kept_limit(int n) { return n / 8 < 1024 ? n / 8 : 1024; }
constexpr int kDirectBodies = 2048;  // colliders of the largest world searched directly
struct SearchRun {
  int direct;
  int fixed_end;
  int cap;
  int may_increment;
};
void launch_search(const DevBodies& b, BroadPhaseBufs& bp, const SearchRun& r, hipStream_t s);
// Where the compaction leaves the pairs: their number, the narrow phase's lists (cuboid-cuboid pairs
// from perm[0] up, the others from perm[pair_cap - 1] down) and their lengths (zeroed by the caller),
// and the manifold index to clear (may be null).
struct PairOut {
  uint32_t* npairs;
  uint32_t* nbox;
  uint32_t* nball;
  uint32_t* perm;
  int* bfirst;
  int pair_cap;
};
size_t compact_tiles(int n);  // tiles of the scan state that the compaction of n bodies takes
// sorted: the segments are in ascending order already
void launch_compact_pairs(const DevBodies& b, BroadPhaseBufs& bp, int cap, bool sorted, const PairOut& o, hipStream_t s);

// k_narrowphase.hip -------------------------------------------------------------------------
struct NarrowPhaseBufs {
  uint32_t* count;        // [P] contacts per pair
  uint32_t* perm;         // [pair_cap] pairs by kind: cuboid-cuboid from the front, the others from the back
  uint32_t* npairs;       // on the device: pairs, cuboid-cuboid pairs, the others
  uint32_t* nbox;
  uint32_t* nball;
  uint32_t* totals;       // [2] contacts (zeroed by the caller), manifolds
  int pair_cap;           // pairs above it are left out (and the caller's to see)
  bool boxes, balls;      // pairs of the kind can occur
  ScanState* scan;
};
// Sorts the first *np.npairs pairs by kind (lists of pairs that did not come from the compaction) and
// clears `out`'s manifold index; nbox and nball are zeroed by the caller.
void launch_narrow_bins(const DevBodies& b, const int2* pairs, NarrowPhaseBufs& np, DevContacts out, hipStream_t s);
size_t manifold_tiles(int npairs);  // tiles of the scan state that the narrow phase takes
void launch_narrow_phase(const DevBodies& b, const int2* pairs, NarrowPhaseBufs& np, DevContacts out, hipStream_t s);
// Contact arrays by row: bodies, feature (as bits), world1, world2, normal, depth (null: not wanted).
struct ContactRows {
  static constexpr int kRows = 6;
  static constexpr int kWidth[kRows] = {2, 1, 3, 3, 3, 1};
  float* row[kRows];
};
// Contact k of manifold m to place moff[m] + k of the rows (at most `cap` places); their number to *counted.
void launch_contacts_out(const DevContacts& c, int M, const uint32_t* moff, uint32_t cap, const ContactRows& out,
                         uint32_t* counted, hipStream_t s);
// Contacts of all manifolds in manifold order, gathered from their slots into dense records
// (kContactFields float4 each) and impulses (dense_imp may be null); moff = exclusive scan of the
// manifolds' counts.
void launch_gather_contacts(const DevContacts& c, int M, const uint32_t* moff, float4* dense,
                            float4* dense_imp, hipStream_t s);

// k_solver.hip -----------------------------------------------------------------------------
struct SolverBufs {
  uint32_t* deg;          // [n] dynamic-body degree in the manifold graph
  uint32_t* adj_off;      // [n]
  int* adj;               // [2M]
  uint2* place;           // [M] place of the manifold in its bodies' lists (kNoPlace: a static body)
  uint32_t* state;        // [M] colouring state: 0xffffffff, or round << 16 | colour
  uint32_t* hist;         // [colour_hist_words] manifolds, then contacts, per colour and tile
  uint32_t* offs;         // [same] their exclusive sums
  uint32_t* ckeys;        // [M] colour of each slot
  uint32_t* col_start;    // [max colours + 1] first slot of each class, and
  uint32_t* class_rec;    // first row record
  int4* sinfo;            // [M] per slot: body1|dyn1<<30, body2|dyn2<<30, first record, count|first<<3
  uint2* slot_of;         // [M] slot and first row record of each manifold
  float4* rec;            // [kRecFields rec_stride] row records, field f of record r at kRecFields r + f
  float4* lam;            // [rec_stride] impulses of each row record (normal, tangent 1, tangent 2) and mu
  float* has;             // [C] 1 where the warm start came from the cache (null: nobody asks)
  float4* prec;           // [3 rec_stride] position records: (lp1 | contact kind), (lp2 | shape 1), (ln | shape 2)
  float4* pgeo;           // [2M] per slot: (half extents 1 | margin 1), (half extents 2 | margin 2)
  long rec_stride;        // record capacity (fixed between reallocations)
  double* red;            // residual partials, in host memory
  uint32_t* tmp;          // radix scratch
  ScanState* scan;
};
constexpr int kMaxColours = 4096;
constexpr int kRecFields = 4;  // float4 per contact row record

// Colours inherited from the previous solve's manifolds, degrees and adjacency (M > 0).
void launch_colour_begin(const DevBodies& b, const DevContacts& c, int M, const DevContacts& prev, int prevM,
                         const uint32_t* prev_state, SolverBufs& sb, hipStream_t s);
// *remaining, zero before, becomes 1 if a manifold stays uncoloured; *last_round the last round that
// coloured one
void launch_colour_round(const DevContacts& c, int M, int round, uint32_t* remaining, uint32_t* last_round,
                         SolverBufs& sb, hipStream_t s);
// Slots, records and classes in colour order; *ncol, zero before, becomes the number of colours. With
// kColourDigits digits and `split`, up to kColourDigits / 2 colours with the manifolds of several contacts first in
// each (class c begins at digits 2 c and 2 c + 1), without it up to `digits` (kColourDigits or kMaxColours) colours.
constexpr int kColourDigits = 512;
size_t colour_hist_words(int M, int digits);
void launch_colour_order(const DevContacts& c, int M, int C, int digits, bool split, SolverBufs& sb, uint32_t* ncol,
                         hipStream_t s);
// All of the above in one launch, for 0 < M <= kSmallManifolds and b.n <= kSmallColourBodies: words[0] becomes 0, words[1]
// too but where a body has too many manifolds for it, which leaves the rounds to launch_colour_round, words[2] the number of colours and words[3] the last round that coloured a manifold. The order is of
// kColourDigits digits, as launch_colour_order's, and where the colours are more it has to be made again.
constexpr int kSmallManifolds = 2048;
constexpr int kSmallColourBodies = 4096;
void launch_colour_small(const DevBodies& b, const DevContacts& c, int M, int C, const DevContacts& prev, int prevM,
                         const uint32_t* prev_state, bool split, SolverBufs& sb, uint32_t* words, hipStream_t s);
int residual_blocks(int M);
void launch_assemble(const DevBodies& b, const DevContacts& cur, const DevContacts& prev,
                     int prevM, int M, const SimParams& p, SolverBufs& sb, const MatTable& mt, hipStream_t s);
// A colour class: its first slot, its manifolds with several contacts (or of any number, where the
// order is not split) and after them those with one.
struct ClassSpan {
  int first, multi, single;
};
// One colour of the warm start and of a sweep.
void launch_warmstart_colour(const DevBodies& b, const ClassSpan& c, SolverBufs& sb, hipStream_t s);
void launch_pgs_colour(const DevBodies& b, const ClassSpan& c, SolverBufs& sb, hipStream_t s,
                       hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);
// Consecutive visited classes, each of at most kRunLanes sweep lanes (8 for a manifold of several contacts, 2
// for one of one), in one workgroup (warm start or sweep). Beyond that a launch of the class's own, on
// many compute units, is faster: velocity solve 254 us against 316 with two or three passes of the workgroup at
// 627 manifolds of 2.7 contacts; with half the lanes 172 us against 155 at 1,233 of one contact, and 406 either way at
// 23,730. Passed by value: no copy to the device stands before the launch.
constexpr int kRunLanes = 1024;
constexpr int kRunClasses = 64;
struct ClassRun {
  int n;
  ClassSpan r[kRunClasses];
};
void launch_colour_run(const DevBodies& b, SolverBufs& sb, const ClassRun& run, bool warm, hipStream_t s);
// cache: also the impulses to the contacts' slots, as launch_cache_impulses
void launch_residual(const DevBodies& b, const DevContacts& c, int M, bool cache, SolverBufs& sb, hipStream_t s);
void launch_cache_impulses(const DevContacts& c, SolverBufs& sb, int M, hipStream_t s);

// Scene-blocked sweeps (k_solver.hip): every scene's slots in (scene, colour) order, per scene
// and colour the first position, and the scene's dynamic bodies (CSR) with each body's rank.
constexpr int kLdsBodies = 2048;  // dynamic bodies of one scene the blocked kernel keeps in LDS
constexpr int kSmallScene = 256;  // scenes up to this many dynamic bodies use the small workgroups
constexpr int kSmallLanes = 128;  // of this many lanes
// Visiting order of the colour classes, by value.
constexpr int kVisitColours = 512;
struct VisitOrder {
  int n, split;
  uint16_t c[kVisitColours];
};
struct SceneBlocks {
  uint32_t* keys;        // [M] scene, sorted
  uint32_t* slot;        // [M] slots in (scene, colour) order; null: the colour order is it (one scene)
  uint32_t* keys_alt;
  uint32_t* slot_alt;
  uint32_t* start;       // [nscenes][digits + 1] (digits: of the colour order, 1 or 2 per colour)
  int4* info;            // [M] the slots' sinfo in that order
  int2* rank;            // [M] and the ranks of their bodies in their scene
  const int* dyn_start;  // [nscenes + 1]
  const int* dyn_list;   // dynamic bodies scene by scene
  const int* local;      // [n] rank of a dynamic body within its scene
  const int* small_list; // scenes with at most kSmallScene dynamic bodies
  const int* large_list; // the other scenes
  int n_small, n_large;
  __device__ int at(int i) const { return slot ? int(slot[i]) : i; }
};
// The class visited k-th, of scene s.
__device__ __forceinline__ ClassSpan scene_span(const SceneBlocks& sc, const VisitOrder& visit, int s, int k) {
  const int per = visit.split ? 2 : 1;
  const uint32_t* st = sc.start + long(s) * (per * visit.n + 1) + per * visit.c[k];
  ClassSpan r;
  r.first = int(st[0]);
  r.multi = int(st[1]) - r.first;
  r.single = visit.split ? int(st[2]) - int(st[1]) : 0;
  return r;
}
void launch_scene_order(const DevBodies& b, int M, int nscenes, int scene_bits, int digits, SolverBufs& sb,
                        SceneBlocks& sc, hipStream_t s);
// block: lanes per large scene (256, 512 or 1024); the large scenes go on s_large, the small on s_small
void launch_sweeps_blocked(const DevBodies& b, SolverBufs& sb, const SceneBlocks& sc, const VisitOrder& visit,
                           int nsweeps, bool warm, int block, hipStream_t s_small, hipStream_t s_large);
// Scene-blocked position correction: `iterations` passes over the colours in the visiting order,
// one workgroup per scene with the scene's dynamic poses in LDS (the same corrections in the same
// order per body as the per-colour launches); streams and block as launch_sweeps_blocked.
void launch_position_blocked(const DevBodies& b, const SimParams& p, SolverBufs& sb, const SceneBlocks& sc,
                             const VisitOrder& visit, int iterations, int block, hipStream_t s_small,
                             hipStream_t s_large);

// learned warm start (k_solver.hip): features [C][24] and impulse units ls [C] per row record,
// the prediction y [C][3] applied as the warm start, post-solve targets t [C][3].
void launch_features(const DevBodies& b, const DevContacts& c, const SimParams& p, int M, SolverBufs& sb, float* X,
                     float* ls, hipStream_t s);
void launch_apply_prediction(SolverBufs& sb, int C, const float* y, const float* ls, hipStream_t s);
void launch_sample_targets(SolverBufs& sb, int C, const float* ls, float* t, hipStream_t s);
void launch_lam_copy(SolverBufs& sb, int C, float4* buf, bool to_buf, hipStream_t s);

// k_joints.hip -----------------------------------------------------------------------------
// Joint constraints (ball, fixed, revolute): static SoA per joint in joint order, a fixed greedy
// colouring (joints sharing a dynamic body differ in colour) with the joints listed colour by
// colour, and per solve one row record per joint at its position in that list.
enum { JOINT_BALL = 0, JOINT_FIXED = 1, JOINT_REVOLUTE = 2, JOINT_PRISMATIC = 3, JOINT_CYLINDRICAL = 4 };
// linear rows of a joint kind (they come first): the prismatic and cylindrical joints' two (the
// directions orthogonal to the axis), the others' three
__host__ __device__ inline int joint_linear_rows(int kind) {
  return kind == JOINT_PRISMATIC || kind == JOINT_CYLINDRICAL ? 2 : 3;
}
constexpr int kJointRec = 10;  // float4 per joint row record
struct JointBufs {
  int nj;                // joints
  int ncol;              // joint colours
  const int4* info;      // [nj] (kind, body1, body2, colour)
  const float4* a1;      // [nj] local anchors
  const float4* a2;
  const float4* f1;      // [nj] fixed: reference frames (i, j, k, w); revolute: local axes (xyz)
  const float4* f2;
  const float2* brk;     // [nj] squared break force, squared break torque
  float4* imp_lin;       // [nj] impulses cached by the last solve
  float4* imp_ang;
  int* state;            // [nj] bit 0 broken, bit 1 removed
  const int* order;      // [nj] joints colour by colour (stable in joint order)
  const int2* crange;    // [ncol] (first position in order, joints)
  // per solve, at the joint's position in `order`: (p1 | rows), (p2 | active), 6 x (dir | r),
  // (rhs 0-3), (rhs 4-5, -, -); impulses of rows 0-3 and 4-5
  float4* rec;
  float4* lam;
};
void launch_joint_assemble(const DevBodies& b, const SimParams& p, JointBufs& j, hipStream_t s);
// one workgroup over every joint colour in order (small joint sets), or one launch per colour
void launch_joint_warm(const DevBodies& b, JointBufs& j, hipStream_t s);
void launch_joint_sweep(const DevBodies& b, JointBufs& j, hipStream_t s);
void launch_joint_position(const DevBodies& b, const SimParams& p, JointBufs& j, hipStream_t s);
void launch_joint_cache(const DevBodies& b, const SimParams& p, JointBufs& j, hipStream_t s);
// residual of the joint rows (phi = w): (max, sum of squares, rows) into out[0..2]
void launch_joint_residual(const DevBodies& b, JointBufs& j, double* out, hipStream_t s);
// union of the bodies of every joint neither broken nor removed (activation islands)
void launch_joint_union(const DevBodies& b, const JointBufs& j, int* parent, uint32_t* touch, hipStream_t s);

// k_ccd.hip --------------------------------------------------------------------------------
struct CcdBufs {
  float* body_time;        // [n] time each body's motion starts from (SubstepState::body_times)
  float* frozen;           // [n] per body key: freeze time, < 0 when not frozen
  int* slot_pair;          // [P] pair index of each CCD slot (pairs with a CCD-enabled side)
  int4* slot_bodies;       // [P] the slot's two bodies and their keys; a key | kSlotStatic when its
                           // body is not dynamic
  // times of impact: key = time bits << 32 | pair index (times are >= 0, so keys order by time, then pair)
  unsigned long long* key;       // [P] each slot's queued one, all ones for none
  unsigned long long* seen_key;  // [2P] per slot and side: with that side's body frozen at seen_at
  float* seen_at;                // [2P] (< 0: not known)
  unsigned long long* group;     // [kCcdGroups] smallest keys of groups of slots, between two launches of the queue
  int* stage;              // [P] slots of one re-sweep to be computed
  int* bodies;             // [n] the dynamic bodies with CCD slots
  unsigned long long* impacts;  // [cap] keys of the confirmed impacts, in order
  uint32_t* ctl;           // control words kCcd*
  int cap;
  uint32_t* in_t;          // [n] per key: its colliders are traversed
  uint32_t* new_t;         // [n] per key: traversed from the next round on
  uint32_t* prep;          // [n] to be moved to its impact time
  uint32_t* prepared;      // [n] moved: the substep's island
  uint32_t* evaluated;     // [P]
  uint32_t* kept;          // [P] manifold not empty at the moved poses
  uint32_t* cand;          // [P] to evaluate in this round
  uint32_t* cpos;          // [P] exclusive scan of a flag array
  int2* list;              // [P] compacted pairs, pair order
  int* list_pair;          // [P] their pair indices
  ScanState* scan;
  uint32_t* deg;           // [n] CCD slots of each dynamic body
  uint32_t* off;           // [n] exclusive scan of deg
  uint32_t* fill;          // [n]
  int* adj;                // [2P] the slots of each dynamic body, at off
};
enum : int {
  kCcdSlots = 0, kCcdBodies = 1, kCcdAnyIn = 2, kCcdMinAfter = 3, kCcdKind = 4, kCcdImpacts = 5,
  kCcdLastToi = 6, kCcdOverflow = 7, kCcdMinOver = 8, kCcdList = 9, kCcdState = 10,
  kCcdWords = 16
};
enum : uint32_t { kQueueNew = 0, kQueueOpen = 1, kQueueDone = 2 };
enum : int { PREDICT_NONE = 0, PREDICT_AFTER_END = 1, PREDICT_IMPACTS = 2 };
constexpr int kCcdGroups = 4096;
constexpr int kSlotStatic = 1 << 30;  // body counts stay below 2^30
// predict_next_impacts up to end_time: control words reset, freeze times cleared and every CCD pair's
// time of impact; then rounds of the queue until ctl[kCcdState] is kQueueDone (kind, impacts and last impact time
// in ctl). A round gets further by one event at least.
void launch_ccd_first(const DevBodies& b, const int2* pairs, int npairs, CcdBufs& c, float end_time, float dt0,
                      float target, int on_penetration, hipStream_t s);
void launch_ccd_events(const DevBodies& b, CcdBufs& c, float end_time, float dt0, float target, int on_penetration,
                       hipStream_t s);
// in_t, new_t, prep and prepared of n, evaluated and kept of P cleared
void launch_ccd_island(int n, int P, CcdBufs& c, hipStream_t s);
void launch_ccd_seed(const DevBodies& b, const int2* pairs, CcdBufs& c, int nimp, hipStream_t s);
void launch_ccd_touch(const DevBodies& b, const int2* pairs, int npairs, CcdBufs& c, hipStream_t s);
void launch_ccd_prepare(const DevBodies& b, CcdBufs& c, float dt_sub, float last_toi, hipStream_t s);
// the pairs with flag[p] != 0 into c.list / c.list_pair in pair order, their count to ctl[kCcdList]
void launch_ccd_compact(const int2* pairs, int npairs, const uint32_t* flag, CcdBufs& c, hipStream_t s);
void launch_ccd_grow(const DevBodies& b, CcdBufs& c, int nlist, const uint32_t* count, hipStream_t s);
void launch_ccd_merge(int n, CcdBufs& c, hipStream_t s);
void launch_ccd_validate(const DevBodies& b, const int2* pairs, CcdBufs& c, int nimp, hipStream_t s);
void launch_ccd_clamp(const DevBodies& b, CcdBufs& c, hipStream_t s);

// k_position.hip ---------------------------------------------------------------------------
void launch_position_colour(const DevBodies& b, const SimParams& p, const ClassSpan& c, SolverBufs& sb,
                            hipStream_t s);
void launch_position_run(const DevBodies& b, const SimParams& p, SolverBufs& sb, const ClassRun& run, hipStream_t s);

}  // namespace nph
