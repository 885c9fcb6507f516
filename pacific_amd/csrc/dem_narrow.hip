// Narrow phase of systems with non-spherical bodies, as kernels of their own:
// for every sorted particle, the closest points of its neighbour candidates
// and of the obstacles (Particle::InterAction, Particle.cpp:477-545, with
// RigidBodyWithCrust::ClosestPoint, RigidBodyWithCrust.cpp:205-354, its GJK
// general path and the ContactError recovery of :534-590; SimpleObstacle::
// InterAction, SimpleObstacle.cpp:222-271), recorded as ContactFeat entries
// in the order of the 27-cell sweep.  The force sweep then reads those
// records, so that the GJK state and the integrator never share a kernel's
// registers.  Contact statistics of the evaluation are collected here.
//
// The work list of the step -- one item per listed candidate a particle
// evaluates and per obstacle whose bounding box it meets -- is written by the
// contact search (k_detect).
//
//   k_narrow_lanes the work list with the default options: a grid of one-wave
//                  workgroups, each lane stepping one distance search and
//                  taking another item when it ends; a contact's record goes
//                  to the item's slot (candidate j: slot j; obstacle o: slot
//                  nc + o)
//   k_narrow_items the work list with other options, and the closed forms
//                  (spheres), one evaluation per lane
//   k_narrow       with contact statistics: one thread per particle over
//                  all its candidates and obstacles, records packed;
//                  through ONE evaluation site (one copy of the GJK state
//                  in registers)
//   k_narrow_full  the particles whose candidates overflowed the list (or
//                  every particle without a list): the generic 27-cell sweep
//
// The force sweep reads slots 0 .. count-1 in order and skips kNoFeat, so
// both layouts give the same contacts in the same order.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dem_device.hpp"
#include "dem_forces.hpp"
#include "dem_launch.hpp"

namespace dem {

// Records each contact (overlap < 0) of one particle.  mirror (k_narrow_full
// beside the work list): the partners with a usable list and a higher id
// make no evaluation of their own of a one-sided pair.
struct FeatureVisitor {
  const ContactFeat& cf;
  int k;
  int c = 0;
  bool mirror = false;
  const Particles* P = nullptr;
  const Sorted* S = nullptr;
  const NbrList* L = nullptr;
  const Self* me = nullptr;
  int s = 0;
  DevStatus* st = nullptr;
  __device__ __forceinline__ void put(int o, int pid, d3 xo, d3 Pc, d3 ov) {
    put_at(c, o, pid, xo, Pc, ov);
    ++c;
  }
  __device__ __forceinline__ void put_at(int slot, int o, int pid, d3 xo, d3 Pc, d3 ov) {
    if (slot < cf.cap) {
      const size_t e = (size_t)slot * cf.n + k;
      cf.ent[e] = o;
      cf.pid[e] = pid;
      cf.f[0][e] = xo.x;
      cf.f[1][e] = xo.y;
      cf.f[2][e] = xo.z;
      cf.f[3][e] = Pc.x;
      cf.f[4][e] = Pc.y;
      cf.f[5][e] = Pc.z;
      cf.f[6][e] = ov.x;
      cf.f[7][e] = ov.y;
      cf.f[8][e] = ov.z;
    }
  }
  static constexpr bool kEager = false;
  __device__ __forceinline__ void pair(int k2, int s2i, int pid2, d3 xo, double, d3 Pc, d3 ov, double d) {
    put(s2i, pid2, xo, Pc, ov);
    if (mirror && pid2 > me->id && L->count[k2] <= L->cap) mirror_full(k2, s2i, pid2, xo, Pc, ov, d);
  }
  __device__ __forceinline__ void mirror_full(int k2, int s2i, int pid2, d3 xo, d3 Pc, d3 ov, double d);
  __device__ __forceinline__ void wall(int o, d3 Pc, d3 ov, double) { put(-1 - o, 0, d3{0., 0., 0.}, Pc, ov); }
};

__device__ __forceinline__ bool load_self(const Particles& P, const Sorted& S, const StepParams& sp, int k, Self& me,
                                          int& s) {
  s = S.order[k];
  if ((unsigned)s >= (unsigned)sp.n) return false;
  const double* pr = S.posr + 4 * (size_t)k;
  me.x = d3{pr[0], pr[1], pr[2]};
  me.r = pr[3];
  me.v = me.w = d3{0., 0., 0.};
  me.m = me.req = 0.;
  me.mat = 0;
  me.id = P.id[s];
  me.c = P.crust[s];
  return true;
}

// A one-sided pair (see one_sided) is evaluated by its lower id, which also
// writes the partner's record -- the mirror image: same point, opposite
// overlap vector -- unless the partner has no usable list (k_narrow_full then
// covers it).  The partner's record slot holds kNoFeat from k_detect until
// then.
__device__ __forceinline__ bool mirrored_pair(const NbrList& L, int code, bool both_spheres, int k2) {
  return one_sided(code, both_spheres) && L.count[k2] <= L.cap;
}

// The slot of body k in its neighbour k2's list (both seen without periodic
// shift; the lists are symmetric: the candidate test is exact under the
// exchange), -1 if it is missing.
__device__ __forceinline__ int slot_in_list(const NbrList& L, int k2, int k) {
  const int nc2 = L.count[k2];
  const unsigned want = nbr_entry(k, 0, 0, 0);
  for (int i0 = 0; i0 < nc2; i0 += 16) {
    unsigned hit = 0u;
#pragma unroll
    for (int u = 0; u < 16; ++u)
      if (i0 + u < nc2 && L.ent[(size_t)(i0 + u) * L.n + k2] == want) hit |= 1u << u;
    if (hit) return i0 + __builtin_ctz(hit);
  }
  return -1;
}

// The record of item j of sorted slot k, and, for a mirrored pair, the
// partner's.
__device__ __forceinline__ void put_item(const StepParams& sp, DevStatus* st, const NbrList& L, int k, int j, int s,
                                         const Self& me, int partner, int pid2, int k2, bool mirror, d3 xo, d3 Pc,
                                         d3 ov) {
  FeatureVisitor vis{sp.cf, k};
  vis.put_at(j, partner, pid2, xo, Pc, ov);
  if (!mirror) return;
  const int jm = slot_in_list(L, k2, k);
  if (jm < 0) {
    raise_error(st, kContactOverflow, me.id, pid2);
  } else {
    FeatureVisitor pv{sp.cf, k2};
    pv.put_at(jm, s, me.id, me.x, Pc, -ov);
  }
}

__device__ __forceinline__ void FeatureVisitor::mirror_full(int k2, int s2i, int pid2, d3 xo, d3 Pc, d3 ov, double d) {
  const double* q2 = S->posr + 4 * (size_t)k2;
  const bool shifted = xo.x != q2[0] || xo.y != q2[1] || xo.z != q2[2];
  const bool both = body_type(*P, s) == kShapeSphere && body_type(*P, s2i) == kShapeSphere;
  if (shifted || both) return;
  const int jm = slot_in_list(*L, k2, k);
  if (jm < 0) {
    raise_error(st, kContactOverflow, me->id, pid2);
    return;
  }
  // a recovered contact (overlap exactly the crusts) counts on both sides
  if (d == -(me->c + P->crust[s2i])) atomicAdd(&st->n_recovered, 1);
  FeatureVisitor pv{cf, k2};
  pv.put_at(jm, s, me->id, me->x, Pc, -ov);
}

// ITEM: the one evaluation `item` of sorted slot k (a listed candidate if
// item < nc, else obstacle item - nc), its record at slot `item`.
// Otherwise: every candidate and obstacle of k, in the order of
// for_each_listed, records packed and counted.  Each evaluation goes
// through the one site below; nothing but the loop state stays live across
// it: both bodies are rebuilt from memory at every pass, and a pair whose
// crust-shrunk bodies intersect comes round once more for the recovery
// (attempt 1).  A particle without a usable list is marked (count -1) for
// k_narrow_full.
// work: the lane's column of the distance search's work area; tab: the shape
// tables.
template <bool ITEM>
__device__ __forceinline__ void narrow_one(const Particles& P, const Sorted& S, const Grid& G,
                                           const BoxObstacle* __restrict__ obs, const StepParams& sp, DevStatus* st,
                                           const NbrList& L, int k, int item, StatAcc* acc, const GjkWork& work,
                                           const ShapeTables& tab) {
  const int cx = sp.cur & 1;
  Self me;
  int s;
  if (!load_self(P, S, sp, k, me, s)) {
    if (!ITEM) sp.cf.count[k] = 0;
    return;
  }
  const int nc = L.count ? L.count[k] : 0;
  if (!L.count || nc > L.cap) {
    if (!ITEM) sp.cf.count[k] = -1;
    return;
  }
  const int self_type = P.shape[s] < 0 ? kShapeSphere : P.shapes[P.shape[s]].type;
  FeatureVisitor vis{sp.cf, k};
  int attempt = 0;
  const int nitems = ITEM ? 1 : nc + sp.nobs;
  for (int it = 0; it < nitems; it += attempt ? 0 : 1) {
    const int j = ITEM ? item : it;
    const int att = attempt;
    attempt = 0;
    d3 Pc, ov, xo{0., 0., 0.};
    double d = 0.;
    int nit = 1, res = 0, partner, pid2, mult;
    int k2 = -1;          // the partner's sorted slot (candidates)
    bool mirror = false;  // this thread also writes the partner's record
    ConvexGeo og;
    bool convex = false;
    if (j < nc) {
      // visit_candidate: periodic image, conservative reject
      const unsigned e = L.ent[(size_t)j * L.n + k];
      k2 = (int)(e & kNbrSlotMask);
      const int code = (int)(e >> kNbrSlotBits);
      const int ix = code % 3 - 1, iy = (code / 3) % 3 - 1, iz = code / 9 - 1;
      const double* q2 = S.posr + 4 * (size_t)k2;
      xo = d3{ix ? q2[0] + image_shift(G, 0, ix) : q2[0], iy ? q2[1] + image_shift(G, 1, iy) : q2[1],
              iz ? q2[2] + image_shift(G, 2, iz) : q2[2]};
      const double ro = q2[3];
      const d3 AB = xo - me.x;
      const double s2 = AB.x * AB.x + AB.y * AB.y + AB.z * AB.z;
      const double R = me.r + ro;
      if (s2 > R * R * 1.000000000001) continue;
      const int s2i = S.order[k2];
      if ((unsigned)s2i >= (unsigned)sp.n) continue;
      partner = s2i;
      pid2 = S.sid[k2];
      const int sh[3] = {ix, iy, iz};
      mult = me.id < pid2 ? image_evaluations(G, me.x, d3{q2[0], q2[1], q2[2]}, sh) : 0;
      const bool osph = P.shape[s2i] < 0 || P.shapes[P.shape[s2i]].type == kShapeSphere;
      if (ITEM && mirrored_pair(L, code, self_type == kShapeSphere && osph, k2)) {
        mirror = true;
      }
      if (self_type == kShapeSphere && osph) {
        const double co = P.crust[s2i];
        res = sphere_sphere(me.x, me.r, me.c, AB, sqrt(s2), ro, co, Pc, ov, d);
        if (res < 0) res = recover_ss(me.x, me.r, me.c, xo, ro, co, Pc, ov, d) ? 2 : -1;
      } else {
        og = convex_of(P, s2i, xo, cx, tab);
        convex = true;
      }
    } else {
      // SimpleObstacle::InterAction: bounding-box pre-test
      const int o = j - nc;
      const BoxObstacle& B = obs[o];
      const bool probable = fabs(B.aabb_c[0] - me.x.x) <= B.aabb_e[0] + me.r &&
                            fabs(B.aabb_c[1] - me.x.y) <= B.aabb_e[1] + me.r &&
                            fabs(B.aabb_c[2] - me.x.z) <= B.aabb_e[2] + me.r;
      if (!probable) continue;
      partner = -1 - o;
      pid2 = B.id;
      mult = 1;
      if (self_type == kShapeSphere) {
        res = sphere_box(B, me.x, me.r, me.c, Pc, ov, d);
        if (res < 0) res = recover_sb(B, me.x, me.r, me.c, Pc, ov, d) ? 2 : -1;
      } else {
        og = convex_of_obstacle(B);
        convex = true;
      }
    }
    if (convex) {
      ConvexGeo mg = convex_of(P, s, me.x, cx, tab);
      mg.work = work;
      // closest_convex: sphere-box closed forms (a closed form that finds
      // the crusts overlapping recovers through GJK), otherwise GJK
      const bool sb = mg.type == kShapeSphere && og.type == kShapeBox;
      const bool bs = mg.type == kShapeBox && og.type == kShapeSphere;
      if ((sb || bs) && att == 0) {
        res = sb ? sphere_box_particle(og, mg, true, Pc, ov, d) : sphere_box_particle(mg, og, false, Pc, ov, d);
        if (res < 0) {
          attempt = 1;
          continue;
        }
      } else {
        res = gjk_attempt(mg, og, att, Pc, ov, d, nit, acc == nullptr);
        if (res < 0 && att == 0) {
          attempt = 1;
          continue;
        }
      }
    }
    if (res == 0) continue;
    if (res < 0) {
      raise_error(st, kContactError, me.id, pid2);
      continue;
    }
    if (res == 2) atomicAdd(&st->n_recovered, mirror ? 2 : 1);  // counted on each body's side
    if (acc && mult) acc->add(d, nit, mult);
    if (!(d < 0.)) continue;
    if (ITEM) {
      put_item(sp, st, L, k, j, s, me, partner, pid2, k2, mirror, xo, Pc, ov);
    } else {
      vis.put(partner, pid2, xo, Pc, ov);
    }
  }
  if (ITEM) return;
  sp.cf.count[k] = vis.c;
  if (vis.c > sp.cf.cap) raise_error(st, kContactOverflow, me.id, vis.c);
}

// Shape classes and polyhedron vertices that a workgroup copies to LDS, so
// that a body's class costs no dependent global load and a support none at
// all; a system with more reads them from memory.
constexpr int kStageShapes = 8;
constexpr int kStageVerts = 64;
struct Staged {
  double verts[3 * kStageVerts];
  ShapeDesc shapes[kStageShapes];
};
struct StagedNone {};
template <bool STAGED>
__device__ __forceinline__ ShapeTables stage_tables(const Particles& P, void* lds) {
  if (!STAGED) return ShapeTables{P.shapes, P.verts};
  Staged* t = (Staged*)lds;
  for (int i = threadIdx.x; i < 3 * P.nverts; i += 64) t->verts[i] = P.verts[i];
  const int words = P.nshapes * (int)(sizeof(ShapeDesc) / 4);
  for (int i = threadIdx.x; i < words; i += 64) ((int*)t->shapes)[i] = ((const int*)P.shapes)[i];
  __syncthreads();
  return ShapeTables{t->shapes, t->verts};
}

// RigidBodyWithCrust::ClosestPoint's closed forms: a sphere with a sphere or
// a box
__device__ __forceinline__ bool closed_pair(int a, int b) {
  return (a == kShapeSphere && b != kShapePoly) || (a == kShapeBox && b == kShapeSphere);
}
__device__ __forceinline__ bool closed_item(const Particles& P, const NarrowItem& it) {
  return closed_pair(body_type(P, it.s), it.partner < 0 ? (int)kShapeBox : body_type(P, it.partner));
}

// The work list one item per lane at a time (one-wave workgroups that stride
// over a part of it each): every item with the signed-volume sub-distance,
// acceleration or a bounding-volume pre-test; with the default options the
// pairs of closed form only (closed), k_narrow_lanes taking the others.
template <bool STAGED>
__global__ __launch_bounds__(64) void k_narrow_items(Particles P, Sorted S, Grid G, const BoxObstacle* __restrict__ obs,
                                                     StepParams sp, DevStatus* st, NbrList L, bool closed) {
  __shared__ double area[kGjkWork * 64];
  __shared__ std::conditional_t<STAGED, Staged, StagedNone> lds;
  const ShapeTables tab = stage_tables<STAGED>(P, &lds);
  const GjkWork W{area + threadIdx.x, 64};
  const int list = blockIdx.x & (kItemLists - 1);
  const NarrowItem* items = sp.cf.items + (size_t)list * sp.cf.item_stride;
  const int total = sp.cf.nitems[list * kItemPad];
  const int stride = (gridDim.x / kItemLists) * 64;
  for (int i = (blockIdx.x / kItemLists) * 64 + threadIdx.x; i < total; i += stride) {
    const NarrowItem it = items[i];
    if (closed && !closed_item(P, it)) continue;
    narrow_one<true>(P, S, G, obs, sp, st, L, it.k, (int)(it.jc & kNbrSlotMask), nullptr, W, tab);
  }
}

// What an evaluation that found a contact (or intersecting bodies) needs
// beside the search, read again from memory so that none of it stays in
// registers during the search.
struct PairItem {
  Self me;
  int pid2, k2;
  bool mirror;
  d3 xo;
};
__device__ __forceinline__ void load_pair(const Particles& P, const Sorted& S, const Grid& G,
                                          const BoxObstacle* __restrict__ obs, const StepParams& sp, const NbrList& L,
                                          const NarrowItem& it, PairItem& q) {
  int s;
  load_self(P, S, sp, it.k, q.me, s);
  q.k2 = -1;
  q.mirror = false;
  q.xo = d3{0., 0., 0.};
  if (it.partner < 0) {
    q.pid2 = obs[-1 - it.partner].id;
    return;
  }
  const int j = (int)(it.jc & kNbrSlotMask), code = (int)(it.jc >> kNbrSlotBits);
  q.k2 = (int)(L.ent[(size_t)j * L.n + it.k] & kNbrSlotMask);
  q.xo = image_of(P, G, it.partner, sp.cur & 1, code);
  q.pid2 = S.sid[q.k2];
  // a pair searched here holds no two spheres
  q.mirror = mirrored_pair(L, code, false, q.k2);
}

// What follows an evaluation: errors, the recovery count, the records.
__device__ __forceinline__ void item_result(const StepParams& sp, DevStatus* st, const NbrList& L,
                                            const NarrowItem& it, const PairItem& q, int res, double d,
                                            d3 Pc, d3 ov) {
  if (res == 0) return;
  if (res < 0) {
    raise_error(st, kContactError, q.me.id, q.pid2);
    return;
  }
  if (res == 2) atomicAdd(&st->n_recovered, q.mirror ? 2 : 1);  // counted on each body's side
  if (d < 0.)
    put_item(sp, st, L, it.k, (int)(it.jc & kNbrSlotMask), it.s, q.me, it.partner, q.pid2, q.k2, q.mirror, q.xo, Pc, ov);
}

// The work list with the default options.  Searches differ in length (most
// pairs are proven apart within a few iterations, the others take up to a
// dozen), so a wave holds up to 64 searches and steps them together; lanes
// whose search has ended take the next items of the wave's run of the list
// as soon as kRefill of them are free (starting a pair costs about as much
// as two iterations, so not at once).  The next items are loaded ahead, so
// that a start waits for one round of loads only.
// Measured on the 200,000-body hopper (343 bodies in a box), per launch: 623
// (68) us with a copy of the search per slot and vertices in memory, 289 (34)
// with one copy over LDS, 232 (35) with the lanes refilled, 171 (30) with the
// items naming what a start loads and the tables in LDS; refilling at 16 as at
// 24 free lanes, 190 us at 40; held to two waves per SIMD the registers spill
// (211 us).  Bound by the latency of one wave per SIMD (296 registers).
constexpr int kRefill = 24;

template <bool STAGED>
__global__ __launch_bounds__(64) void k_narrow_lanes(Particles P, Sorted S, Grid G, const BoxObstacle* __restrict__ obs,
                                                     StepParams sp, DevStatus* st, NbrList L) {
  __shared__ double area[kGjkWork * 64];
  __shared__ std::conditional_t<STAGED, Staged, StagedNone> lds;
  const ShapeTables tab = stage_tables<STAGED>(P, &lds);
  const GjkWork W{area + threadIdx.x, 64};
  const int cx = sp.cur & 1;
  const int lane = threadIdx.x;
  const int list = blockIdx.x & (kItemLists - 1), waves = gridDim.x / kItemLists;
  const NarrowItem* items = sp.cf.items + (size_t)list * sp.cf.item_stride;
  const int total = sp.cf.nitems[list * kItemPad];
  const int per = (total + waves - 1) / waves;
  int next = (int)(blockIdx.x / kItemLists) * per;
  const int end = min(next + per, total);
  auto ahead = [&]() { return next + lane < end ? items[next + lane] : NarrowItem{0, 0u, 0, 0}; };
  NarrowItem pre = ahead();
  bool active = false;
  NarrowItem it{0, 0u, 0, 0};
  int att = 0;
  ConvexGeo A{}, B{};
  Tf a2w{}, b2w{};
  GjkState g{};
  double crusts = 0.;
  auto start = [&]() {
    const double* pr = S.posr + 4 * (size_t)it.k;
    A = convex_of(P, it.s, d3{pr[0], pr[1], pr[2]}, cx, tab);
    A.opt.sv = A.opt.accel = A.opt.bv = 0;
    if (it.partner >= 0) B = convex_of(P, it.partner, image_of(P, G, it.partner, cx, (int)(it.jc >> kNbrSlotBits)), cx, tab);
    else B = convex_of_obstacle(obs[-1 - it.partner]);
    crusts = A.crust + B.crust;
    // closed forms are k_narrow_items'; one with intersecting bodies as well
    active = !closed_pair(A.type, B.type) && gjk_frames(A, B, att, a2w, b2w);
    if (active) gjk_begin(A, a2w, B, b2w, g);
  };
  for (;;) {
    const unsigned long long idle = __ballot(!active);
    const int nidle = __popcll(idle);
    if (next < end && nidle >= kRefill) {
      // the r-th free lane takes the r-th of the items loaded ahead
      const int r = __popcll(idle & ((1ull << lane) - 1ull));
      const NarrowItem mine{__shfl(pre.k, r), (unsigned)__shfl((int)pre.jc, r), __shfl(pre.s, r), __shfl(pre.partner, r)};
      const bool got = !active && next + r < end;
      next += nidle;
      pre = ahead();
      if (got) {
        it = mine;
        att = 0;
        // (a body whose candidates overflowed its list is k_narrow_full's)
        if (L.count[it.k] <= L.cap) start();
      }
      continue;
    }
    if (nidle == 64) break;
    if (active) {
      const int go = gjk_step(A, a2w, B, b2w, W, att == 0 ? crusts : -1., g);
      if (go == 2) active = false;
      if (go == 0) {
        d3 pa, pb, Pc, ov;
        double d = 0.;
        j_points(W, g.bits, pa, pb);
        const int res = gjk_features(a2w, b2w, att, crusts, g.dist, pa, pb, Pc, ov, d);
        active = false;
        if (res < 0 && att == 0) {
          att = 1;
          start();
        } else if (res != 1 || d < 0.) {
          PairItem q;
          load_pair(P, S, G, obs, sp, L, it, q);
          item_result(sp, st, L, it, q, res, d, Pc, ov);
        }
      }
    }
  }
}

// The generic 27-cell sweep for the particles k_narrow marked.
__device__ __forceinline__ void narrow_full_one(const Particles& P, const Sorted& S, const Grid& G,
                                                const BoxObstacle* __restrict__ obs, const StepParams& sp,
                                                DevStatus* st, const NbrList& L, int k, StatAcc* acc,
                                                const GjkWork& work, bool mirror) {
  const int cx = sp.cur & 1;
  Self me;
  int s;
  if (!load_self(P, S, sp, k, me, s)) return;
  me.acc = acc;
  ConvexGeo mg = convex_of(P, s, me.x, cx, ShapeTables{P.shapes, P.verts});
  mg.work = work;
  FeatureVisitor vis{sp.cf, k};
  vis.mirror = mirror;
  vis.P = &P;
  vis.S = &S;
  vis.L = &L;
  vis.me = &me;
  vis.s = s;
  vis.st = st;
  for_each_contact<FeatureVisitor, true>(P, S, G, obs, sp.nobs, st, 0, 0, sp.n, k, me, vis, &mg, cx);
  sp.cf.count[k] = vis.c;
  if (vis.c > sp.cf.cap) raise_error(st, kContactOverflow, me.id, vis.c);
}

// One thread per sorted slot, records packed: with statistics (256-thread
// workgroups whose partial sums k_stats_fold adds up), and for lists too
// long for the slot layout.
// (BS threads: 256 with statistics)
template <int BS>
__global__ __launch_bounds__(BS) void k_narrow(Particles P, Sorted S, Grid G, const BoxObstacle* __restrict__ obs,
                                               StepParams sp, DevStatus* st, NbrList L) {
  __shared__ double area[kGjkWork * BS];
  const GjkWork W{area + threadIdx.x, BS};
  const int k = xcd_tile(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  const bool mine = k < sp.n && !st->code;  // an error ended the run
  if (BS == 64) {
    if (mine) narrow_one<false>(P, S, G, obs, sp, st, L, k, 0, nullptr, W, ShapeTables{P.shapes, P.verts});
    return;
  }
  StatAcc acc;
  if (mine) narrow_one<false>(P, S, G, obs, sp, st, L, k, 0, &acc, W, ShapeTables{P.shapes, P.verts});
  block_stats(acc, sp.stats + 5 * (size_t)blockIdx.x);
}

template <int BS>
__global__ __launch_bounds__(BS) void k_narrow_full(Particles P, Sorted S, Grid G,
                                                    const BoxObstacle* __restrict__ obs, StepParams sp,
                                                    DevStatus* st, NbrList L, bool mirror) {
  // the work list is empty again for the next step
  if (blockIdx.x == 0 && threadIdx.x < kItemLists) sp.cf.nitems[threadIdx.x * kItemPad] = 0;
  __shared__ double area[kGjkWork * BS];
  const GjkWork W{area + threadIdx.x, BS};
  const int k = xcd_tile(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  const bool mine = k < sp.n && sp.cf.count[k] < 0 && !st->code;
  if (BS == 64) {
    if (mine) narrow_full_one(P, S, G, obs, sp, st, L, k, nullptr, W, mirror);
    return;
  }
  StatAcc acc;
  if (mine) narrow_full_one(P, S, G, obs, sp, st, L, k, &acc, W, false);
  block_stats<true>(acc, sp.stats + 5 * (size_t)blockIdx.x);
}

hipError_t launch_narrow(const Particles& P, const Sorted& S, const Grid& G, const BoxObstacle* obs,
                         const StepParams& sp, DevStatus* st, const NbrList& L, hipStream_t stream) {
  if (sp.n == 0) return hipSuccess;
  const dim3 grid64((sp.n + 63) / 64), grid256((sp.n + 255) / 256);
  // packed records where slots would not fit the obstacles' records
  if (sp.stats) {
    hipLaunchKernelGGL(k_narrow<256>, grid256, dim3(256), 0, stream, P, S, G, obs, sp, st, L);
    hipLaunchKernelGGL(k_narrow_full<256>, grid256, dim3(256), 0, stream, P, S, G, obs, sp, st, L, false);
    return hipGetLastError();
  }
  if (!L.count || L.cap + sp.nobs > sp.cf.cap) {
    hipLaunchKernelGGL(k_narrow<64>, grid64, dim3(64), 0, stream, P, S, G, obs, sp, st, L);
    hipLaunchKernelGGL(k_narrow_full<64>, grid64, dim3(64), 0, stream, P, S, G, obs, sp, st, L, false);
    return hipGetLastError();
  }
  const dim3 grid(sp.cf.item_blocks), block(64);
  const bool plain = !P.gjk.sv && !P.gjk.accel && !P.gjk.bv;
  const bool staged = P.nverts <= kStageVerts && P.nshapes <= kStageShapes;
  if (plain) {
    if (staged) hipLaunchKernelGGL(k_narrow_lanes<true>, grid, block, 0, stream, P, S, G, obs, sp, st, L);
    else hipLaunchKernelGGL(k_narrow_lanes<false>, grid, block, 0, stream, P, S, G, obs, sp, st, L);
  }
  if (!plain || P.spheres) {
    if (staged) hipLaunchKernelGGL(k_narrow_items<true>, grid, block, 0, stream, P, S, G, obs, sp, st, L, plain);
    else hipLaunchKernelGGL(k_narrow_items<false>, grid, block, 0, stream, P, S, G, obs, sp, st, L, plain);
  }
  hipLaunchKernelGGL(k_narrow_full<64>, grid64, block, 0, stream, P, S, G, obs, sp, st, L, true);
  return hipGetLastError();
}

}  // namespace dem
