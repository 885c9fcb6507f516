// HIP kernels of the Grains3D DEM time step for gfx950 (MI355X).
//
// Per step (SecondOrderLeapFrog, kick-drift-kick, Grains.cpp:344-364):
//   k_move / fused tail  half kick + drift + quaternion update, periodic role
//                        swap, cell key, atomic per-cell arrival slot
//   k_scan_*             exclusive prefix of the per-cell counts -> start[]
//   k_scatter            storage index to (cell, arrival slot)
//   k_canon              per particle: its rank by id in its cell, (x,y,z,r)
//                        into the sorted tile array
//   k_detect             a few lanes per sorted particle: 27-cell sweep with
//                        minimum-image shifts, neighbour candidates -> list
//   k_forces<MODE>       one thread per particle (storage order; sorted order
//                        with non-spherical bodies): the listed (or, with no
//                        list, the 27-cell) candidates with
//                        minimum-image shifts, sphere-sphere / sphere-box
//                        closest points, Hooke-dashpot-Coulomb force and
//                        torque gathered in registers (no atomics), then the
//                        second half kick, optionally fused with the next
//                        step's first half kick and drift.
//
// FP64 arithmetic follows the reference expression order and the library is
// built with -ffp-contract=off; the mixed kernels evaluate the force model in
// FP32 (contact decisions stay FP64 so the contact list is identical).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>

#include "dem_device.hpp"
#include "dem_forces.hpp"
#include "dem_launch.hpp"

namespace dem {

// list entries in flight per particle (2: the same, 1: 33 us instead of 30.6 for the 1M gas)
constexpr int kFilterGroup = 4;

// ---------------------------------------------------------------------------
// First half kick + drift over storage indices (in place): Grains.cpp:353
// moveParticlesAndObstacles(dt/2, dt, dt) -> AllComponents::Move.
__global__ __launch_bounds__(256) void k_move(Particles P, Sorted S, Grid G, StepParams sp, DevStatus* st,
                                              double dtv, double dtx, VerletState V, int number) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  // the number of these positions (DevStatus::seq); no list rebuild is under
  // way: both sets of its counters start anew
  if (V.stamp > 0 && s == 0) {
    st->seq[sp.cur & 1] = number;
    st->stop[sp.cur & 1] = st->code != 0;
  }
  if (V.sync && s < 2 * (int)(sizeof(RebuildSync) / sizeof(int))) ((int*)V.sync)[s] = 0;
  if (s >= sp.n) return;
  const int cx = sp.cur & 1, cv = (sp.cur >> 1) & 1;
  Kin k = load_kin(P, s, cx, cv);
  d3 F = ld3(P.F, s), T = ld3(P.T, s);
  double mass = P.mass[s], cf = P.cfac[s], I = P.inertia[s];
  double depl;
  if (P.shape) {
    // system with non-spherical particles (LeapFrog only): basis in place
    double B[9];
    for (int j = 0; j < 9; ++j) B[j] = P.B[cx][j][s];
    const int sh = P.shape[s];
    const bool gyro = sh >= 0 && P.shapes[sh].type != kShapeSphere;
    const d3 I3 = gyro ? d3{P.I3[0][s], P.I3[1][s], P.I3[2][s]} : d3{I, I, I};
    depl = lf_move_body(k, gyro, F, T, mass, cf, I, I3, dtv, dtx, B);
    for (int j = 0; j < 9; ++j) P.B[cx][j][s] = B[j];
  } else if (sp.scheme == kLeapFrog) {
    depl = lf_move(k, F, T, mass, cf, I, dtv, dtx);
  } else {
    AB2State ab;
    if (sp.scheme == kAdamsBashforth2) {
      ab.v_nm2 = ld3(P.v_nm2, s);
      ab.dUdt_nm2 = ld3(P.dUdt_nm2, s);
      ab.wb_nm2 = ld3(P.wb_nm2, s);
      ab.dWdt_nm2 = ld3(P.dWdt_nm2, s);
    }
    depl = other_move(sp.scheme, sp.first_step != 0, k, ab, F, T, mass, cf, I, dtv, dtx);
    if (sp.scheme == kAdamsBashforth2) {
      st3(P.v_nm2, s, ab.v_nm2);
      st3(P.dUdt_nm2, s, ab.dUdt_nm2);
      st3(P.wb_nm2, s, ab.wb_nm2);
      st3(P.dWdt_nm2, s, ab.dWdt_nm2);
    }
  }
  if (depl > P.crust[s]) raise_error(st, kMotionError, P.id[s], 0);  // Particle.cpp:444-456
  wrap_and_bin(k, G, S, st, s, P.id, 0, &V, cx, number + 1);
  st3(P.x[cx], s, k.x);
  st3(P.v[cv], s, k.v);
  st3(P.w[cv], s, k.w);
  st3(P.wb, s, k.wb);
  P.q[0][s] = k.q.v.x;
  P.q[1][s] = k.q.v.y;
  P.q[2][s] = k.q.v.z;
  P.q[3][s] = k.q.w;
}

// Cell key and arrival slot of the current positions, without motion (used
// after initialisation and after a state upload).  Positions outside the
// periodic box are brought back first.
__global__ __launch_bounds__(256) void k_key(Particles P, Sorted S, Grid G, StepParams sp, DevStatus* st,
                                             VerletState V) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= sp.n) return;
  const int cx = sp.cur & 1, cv = (sp.cur >> 1) & 1;
  Kin k = load_kin(P, s, cx, cv);
  d3 x0 = k.x;
  // with a Verlet list the periodic wrap only (the list is rebuilt next)
  wrap_and_bin(k, G, S, st, s, P.id, 0, &V);
  if (k.x.x != x0.x || k.x.y != x0.y || k.x.z != x0.z) {
    st3(P.x[cx], s, k.x);
    st3(P.wb, s, k.wb);
  }
}

// ---------------------------------------------------------------------------
// Exclusive scan of the per-cell counts.  Tiles of 256 threads x 8 cells.
constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ __forceinline__ int block_exclusive_scan(int v, int* lds, int& total) {
  // Hillis-Steele over 256 entries in LDS
  int t = threadIdx.x;
  lds[t] = v;
  __syncthreads();
  for (int off = 1; off < kScanThreads; off <<= 1) {
    int add = t >= off ? lds[t - off] : 0;
    __syncthreads();
    lds[t] += add;
    __syncthreads();
  }
  int incl = lds[t];
  total = lds[kScanThreads - 1];
  __syncthreads();
  return incl - v;
}

// A thread's kScanItems consecutive cells at c0 (a multiple of kScanItems, in
// arrays as aligned as device allocations are): two 16-byte accesses, but for
// the last cells of the grid.
__device__ __forceinline__ void load_cells(const int* __restrict__ a, int c0, int ncells, int (&v)[kScanItems]) {
  if (c0 + kScanItems <= ncells) {
    const int4 lo = *(const int4*)(a + c0), hi = *(const int4*)(a + c0 + 4);
    v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
    v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
  } else {
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) v[i] = c0 + i < ncells ? a[c0 + i] : 0;
  }
}
__device__ __forceinline__ void store_cells(int* __restrict__ a, int c0, int ncells, const int (&v)[kScanItems]) {
  if (c0 + kScanItems <= ncells) {
    *(int4*)(a + c0) = int4{v[0], v[1], v[2], v[3]};
    *(int4*)(a + c0 + 4) = int4{v[4], v[5], v[6], v[7]};
  } else {
#pragma unroll
    for (int i = 0; i < kScanItems; ++i)
      if (c0 + i < ncells) a[c0 + i] = v[i];
  }
}

__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(const int* __restrict__ count, int ncells,
                                                              int* __restrict__ block_sums, const int* gate,
                                                              const int* seq) {
  if (gate && *gate != *seq + 1) return;  // Verlet list still valid: nothing to rebuild
  __shared__ int lds[kScanThreads];
  int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  int vals[kScanItems], sum = 0;
  load_cells(count, base, ncells, vals);
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) sum += vals[i];
  int total;
  block_exclusive_scan(sum, lds, total);
  if (threadIdx.x == 0) block_sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(kScanThreads) void k_scan_top(int* __restrict__ block_sums, int nblocks, const int* gate,
                                                           const int* seq) {
  if (gate && *gate != *seq + 1) return;  // Verlet list still valid: nothing to rebuild
  __shared__ int lds[kScanThreads];
  int carry = 0;
  for (int b0 = 0; b0 < nblocks; b0 += kScanThreads) {
    int i = b0 + threadIdx.x;
    int v = i < nblocks ? block_sums[i] : 0;
    int total;
    int ex = block_exclusive_scan(v, lds, total);
    if (i < nblocks) block_sums[i] = ex + carry;
    carry += total;
  }
}

// FOLD: block_sums holds the tiles' totals (no k_scan_top launch) and each
// block adds those before it itself -- for grids of at most kScanFoldTiles
// tiles, where the sums are cheaper than a launch.
constexpr int kScanFoldTiles = 4096;

// The counts are read here for the last time and cleared for the next binning.
template <bool FOLD>
__global__ __launch_bounds__(kScanThreads) void k_scan_down(int* __restrict__ count, int ncells,
                                                            const int* __restrict__ block_sums,
                                                            int* __restrict__ start, int n, const int* gate,
                                                            const int* seq) {
  if (gate && *gate != *seq + 1) return;  // Verlet list still valid: nothing to rebuild
  __shared__ int lds[kScanThreads];
  int offset;
  if (FOLD) {
    int part = 0;
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += kScanThreads) part += block_sums[b];
    block_exclusive_scan(part, lds, offset);
  } else {
    offset = block_sums[blockIdx.x];
  }
  int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  int vals[kScanItems];
  int sum = 0;
  load_cells(count, base, ncells, vals);
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) sum += vals[i];
  int total;
  int run = block_exclusive_scan(sum, lds, total) + offset;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    const int v = vals[i];
    vals[i] = run;
    run += v;
  }
  store_cells(start, base, ncells, vals);
  const int zero[kScanItems] = {};
  store_cells(count, base, ncells, zero);
  if (blockIdx.x == 0 && threadIdx.x == 0) start[ncells] = n;
}

// Storage index -> (cell start + arrival slot)
__global__ __launch_bounds__(256) void k_scatter(Sorted S, int n, const int* gate, const int* seq) {
  if (gate && *gate != *seq + 1) return;  // Verlet list still valid: nothing to rebuild
  for (int s = blockIdx.x * blockDim.x + threadIdx.x; s < n; s += gridDim.x * blockDim.x) {
    int dst = S.start[S.key[s]] + S.slot[s];
    if ((unsigned)dst < (unsigned)n) S.tmp_order[dst] = s;
  }
}

// One thread per particle: its rank by id in its cell (rank_particle).
// Measured per launch against a thread per cell that sorted its particles: 343
// polyhedra 17.7 -> 5.7 us, 810,527 spheres of a batch 43 -> 24 us.
__global__ __launch_bounds__(256) void k_canon(Particles P, Sorted S, int cx, int n, const int* gate, const int* seq) {
  if (gate && *gate != *seq + 1) return;  // Verlet list still valid: nothing to rebuild
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x)
    rank_particle(P, S, j, cx, n);
}

// ---------------------------------------------------------------------------
// Broad phase of one step (LinkedCell::ComputeForces, LinkedCell.cpp:1019-1103):
// every neighbour candidate of each sorted particle that passes the
// conservative distance reject of the narrow phase, in the order the force
// sweep visits them, written to the candidate list; the force sweep then reads
// a short list instead of 27 cells.  LANES lanes share a particle and test that
// many consecutive candidates at once (the accepted ones numbered by a ballot):
// one lane alone waits for its candidates' loads one after the other, which few
// particles have nothing to fill with (46.8 us per launch for 343 polyhedra,
// whose 27 cells hold about 96 bodies each; 21.6 us with eight, work list
// included; a launch of its own wrote the work list of 200,000 in 59 us).  The
// rule and its figures stand at launch_detect.
// ITEMS (systems with non-spherical bodies): each listed slot's contact
// record starts as kNoFeat, so that the narrow phase writes only contacts, and
// the evaluations the narrow phase has to make are appended to its work list:
// one for each candidate unless the partner's side makes it (a pair without
// periodic shift is evaluated once, by its lower id, see mirrored_pair) and
// one for each obstacle whose bounding box the particle meets.
// After an error raised on the device (which ends the run) the contact
// searches return at once, so that the rest of a batch of steps costs
// little whatever the state has become.
constexpr int kItemBuf = 1024;  // items a workgroup collects before it appends them

template <bool ITEMS, int LANES>
__global__ __launch_bounds__(kDetectThreads) void k_detect(Particles P, Sorted S, Grid G,
                                                                         const BoxObstacle* __restrict__ obs,
                                                                         StepParams sp, NbrList L,
                                                                         const DevStatus* st) {
  __shared__ NarrowItem buf[ITEMS ? kItemBuf : 1];
  __shared__ int nbuf, base;
  if (st->code) return;
  const int n = sp.n;
  const int lane = threadIdx.x & (LANES - 1);
  const int gshift = threadIdx.x & 63 & ~(LANES - 1);
  const int k = xcd_tile(blockIdx.x, gridDim.x) * (kDetectThreads / LANES) + threadIdx.x / LANES;
  if (ITEMS) {
    if (threadIdx.x == 0) nbuf = 0;
    __syncthreads();
  }
  const int list = blockIdx.x & (kItemLists - 1);
  NarrowItem* const items = ITEMS ? sp.cf.items + (size_t)list * sp.cf.item_stride : nullptr;
  int* const nitems = ITEMS ? sp.cf.nitems + list * kItemPad : nullptr;
  if (k < n) {
    const double* pr = S.posr + 4 * (size_t)k;
    const d3 x{pr[0], pr[1], pr[2]};
    const double r = pr[3];
    const int s = ITEMS ? S.order[k] : 0;
    const bool body = !ITEMS || (unsigned)s < (unsigned)n;
    const int id = ITEMS && body ? P.id[s] : 0;
    const bool sphere = ITEMS && P.spheres && body && body_type(P, s) == kShapeSphere;
    auto append = [&](unsigned jc, int partner) {
      const NarrowItem it{k, jc, s, partner};
      const int i = atomicAdd(&nbuf, 1);
      if (i < kItemBuf) buf[i] = it;
      else items[atomicAdd(nitems, 1)] = it;
    };
    int c = 0;
    if constexpr (LANES == 1 && !ITEMS) {
      // one candidate at a time: at this register count eight waves per SIMD
      // overlap the loads better than wider batches of loads per thread do
      for_each_candidate(S, G, 0, 0, n, x, [&](int k2, int ix, int iy, int iz) {
        if (k2 == k) return;
        const double* q2 = S.posr + 4 * (size_t)k2;
        const d3 xo{ix ? q2[0] + image_shift(G, 0, ix) : q2[0], iy ? q2[1] + image_shift(G, 1, iy) : q2[1],
                    iz ? q2[2] + image_shift(G, 2, iz) : q2[2]};
        const d3 AB = xo - x;
        const double s2 = AB.x * AB.x + AB.y * AB.y + AB.z * AB.z;
        const double R = r + q2[3];
        if (s2 > R * R * 1.000000000001) return;
        if (c < L.cap) L.ent[(size_t)c * n + k] = nbr_entry(k2, ix, iy, iz);
        ++c;
      });
      L.count[k] = c;
      return;
    }
    for_each_run(S, G, 0, 0, n, x, [&](int b, int e, int ix, int iy, int iz) {
      for (int k0 = b; k0 < e; k0 += LANES) {
        const int k2 = k0 + lane;
        bool hit = k2 < e && k2 != k;
        if (hit) {
          const double* q2 = S.posr + 4 * (size_t)k2;
          const d3 xo{ix ? q2[0] + image_shift(G, 0, ix) : q2[0], iy ? q2[1] + image_shift(G, 1, iy) : q2[1],
                      iz ? q2[2] + image_shift(G, 2, iz) : q2[2]};
          const d3 AB = xo - x;
          const double s2 = AB.x * AB.x + AB.y * AB.y + AB.z * AB.z;
          const double R = r + q2[3];
          hit = !(s2 > R * R * 1.000000000001);
        }
        const unsigned hits = LANES == 1 ? (unsigned)hit : (unsigned)(__ballot(hit) >> gshift) & ((1u << LANES) - 1u);
        const int j = c + __popc(hits & ((1u << lane) - 1u));
        if (hit && j < L.cap) {
          const unsigned e2 = nbr_entry(k2, ix, iy, iz);
          L.ent[(size_t)j * n + k] = e2;
          if (ITEMS) {
            sp.cf.ent[(size_t)j * n + k] = kNoFeat;
            const int o = S.order[k2];
            if (body && (unsigned)o < (unsigned)n) {
              const bool both = sphere && body_type(P, o) == kShapeSphere;
              const int code = (int)(e2 >> kNbrSlotBits);
              if (!(one_sided(code, both) && id > S.sid[k2])) append((unsigned)j | (e2 & ~kNbrSlotMask), o);
            }
          }
        }
        c += __popc(hits);
      }
    });
    if (lane == 0) L.count[k] = c;
    if (ITEMS) {
      int last = -1;
      if (body && c <= L.cap)
        for (int o0 = 0; o0 < sp.nobs; o0 += LANES) {
          const int o = o0 + lane;
          bool met = false;
          if (o < sp.nobs) {
            const BoxObstacle& B = obs[o];
            met = fabs(B.aabb_c[0] - x.x) <= B.aabb_e[0] + r && fabs(B.aabb_c[1] - x.y) <= B.aabb_e[1] + r &&
                  fabs(B.aabb_c[2] - x.z) <= B.aabb_e[2] + r;
          }
          const unsigned hits = LANES == 1 ? (unsigned)met : (unsigned)(__ballot(met) >> gshift) & ((1u << LANES) - 1u);
          if (met && c + o < sp.cf.cap) append((unsigned)(c + o) | ((unsigned)kNbrNoShift << kNbrSlotBits), -1 - o);
          if (hits) last = o0 + 31 - __builtin_clz(hits);
        }
      // every obstacle slot the force sweep will read, met or not, starts empty
      for (int o = lane; o <= last; o += LANES)
        if (c + o < sp.cf.cap) sp.cf.ent[(size_t)(c + o) * n + k] = kNoFeat;
      // a body without a usable list: -1, k_narrow_full searches its cells
      if (lane == 0) sp.cf.count[k] = !body ? 0 : (c > L.cap ? -1 : c + last + 1);
    }
  }
  if (ITEMS) {
    __syncthreads();
    const int m = min(nbuf, kItemBuf);
    if (threadIdx.x == 0) base = m ? atomicAdd(nitems, m) : 0;
    __syncthreads();
    for (int i = threadIdx.x; i < m; i += kDetectThreads) items[base + i] = buf[i];
  }
}

// ---------------------------------------------------------------------------
// Force sweep.  MODE: 0 forces only; 1 forces + second half kick; 2 forces +
// second half kick + next step's Move (LeapFrog) or forces + Move(dt, dt)
// (the other schemes).
// Running totals of the contact statistics after a force launch of nb
// blocks: tot = {overlap sum, overlap max, time of the max, contacts, GJK
// iterations, evaluations with iterations}; the maximum keeps the first
// time it was reached (AppCollision.cpp:174-178).
__global__ __launch_bounds__(256) void k_stats_fold(const double* __restrict__ part, int nb, double* tot,
                                                    double time) {
  StatAcc a;
  for (int i = threadIdx.x; i < nb; i += blockDim.x) {
    const double* p = part + 5 * (size_t)i;
    a.sum += p[0];
    a.max = fmax(a.max, p[1]);
    a.cnt += p[2];
    a.git += p[3];
    a.gn += p[4];
  }
  __shared__ double r[5];
  block_stats(a, r);
  __syncthreads();
  if (threadIdx.x == 0) {
    tot[0] += r[0];
    if (r[1] > tot[1]) {
      tot[1] = r[1];
      tot[2] = time;
    }
    tot[3] += r[2];
    tot[4] += r[3];
    tot[5] += r[4];
  }
}

hipError_t launch_stats_fold(const double* part, int n, double* tot, double time, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_stats_fold, dim3(1), dim3(256), 0, stream, part, (n + 255) / 256, tot, time);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Contacts of a step with the Verlet list: the listed candidates of each
// sphere that pass the narrow phase's conservative distance reject at the
// current positions, in the list's order.  Few registers, so that many
// waves overlap the dependent loads of the list; the force sweep then
// visits only these pairs (same pairs, same order, same arithmetic).
__global__ __launch_bounds__(256) void k_vfilter(Particles P, Sorted S, Grid G, VerletState VS, int n, int cx,
                                                 NbrList L, NbrList CL, TouchList TL, DevStatus* st) {
  __shared__ int nbuf[4], base;
  const int s = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (st->code) return;
  const bool mine = s < n;
  const d3 x = mine ? ld3(P.x[cx], s) : d3{0., 0., 0.};
  const double r = mine ? P.rad[s] : 0.;
  int c2 = 0;
  auto touches = [&](const d3& x2, double r2) {
    const d3 xo = nearest_image(G, x2, x);
    const d3 AB = xo - x;
    const double s2 = AB.x * AB.x + AB.y * AB.y + AB.z * AB.z;
    const double R = r + r2;
    return !(s2 > R * R * 1.000000000001);
  };
  auto keep = [&](int s2i) {
    if (c2 < CL.cap) CL.ent[(size_t)c2 * n + s] = (unsigned)s2i;
    ++c2;
  };
  const int c = mine ? L.count[s] : 0;
  if (c <= L.cap) {
    // a few entries at a time: their loads, and then the neighbours', overlap
    for (int i0 = 0; i0 < c; i0 += kFilterGroup) {
      unsigned e[kFilterGroup];
      d3 x2[kFilterGroup];
      double r2[kFilterGroup];
#pragma unroll
      for (int u = 0; u < kFilterGroup; ++u) e[u] = i0 + u < c ? L.ent[(size_t)(i0 + u) * L.n + s] : ~0u;
#pragma unroll
      for (int u = 0; u < kFilterGroup; ++u) {
        const int o = e[u] < (unsigned)n ? (int)e[u] : s;
        x2[u] = d3{P.x[cx][0][o], P.x[cx][1][o], P.x[cx][2][o]};
        r2[u] = P.rad[o];
      }
#pragma unroll
      for (int u = 0; u < kFilterGroup; ++u)
        if (e[u] < (unsigned)n && touches(x2[u], r2[u])) keep((int)e[u]);
    }
  } else {
    const d3 xb{VS.xb[0][s], VS.xb[1][s], VS.xb[2][s]};
    for_each_candidate(S, VS.Gv, 0, 0, n, xb, [&](int k2, int, int, int) {
      const int s2i = S.order[k2];
      if (s2i != s && (unsigned)s2i < (unsigned)n &&
          touches(d3{P.x[cx][0][s2i], P.x[cx][1][s2i], P.x[cx][2][s2i]}, P.rad[s2i]))
        keep(s2i);
    });
  }
  if (TL.idx) {
    // appended with one atomic per workgroup, in storage order within it
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned long long m = __ballot(c2 != 0);
    if (lane == 0) nbuf[w] = __popcll(m);
    __syncthreads();
    const int list = blockIdx.x & (kTouchLists - 1);
    if (threadIdx.x == 0) {
      const int t = nbuf[0] + nbuf[1] + nbuf[2] + nbuf[3];
      base = t ? atomicAdd(TL.count + list * kItemPad, t) : 0;
    }
    __syncthreads();
    int at = base + __popcll(m & ((1ull << lane) - 1ull));
    for (int k = 0; k < w; ++k) at += nbuf[k];
    if (c2 != 0) TL.idx[(size_t)list * TL.stride + at] = s;
  }
  if (mine) CL.count[s] = c2;
}

// ---------------------------------------------------------------------------
// Host-side launchers
static inline int nblk(int n, int b) { return (n + b - 1) / b; }

hipError_t launch_move(const Particles& P, const Sorted& S, const Grid& G, const StepParams& sp, DevStatus* st,
                       double dtv, double dtx, const VerletState& V, int number, hipStream_t stream) {
  if (sp.n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_move, dim3(nblk(sp.n, 256)), dim3(256), 0, stream, P, S, G, sp, st, dtv, dtx, V, number);
  return hipGetLastError();
}

__global__ void k_clear_ints(int* p, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

hipError_t launch_clear(int* p, int n, hipStream_t stream) {
  hipLaunchKernelGGL(k_clear_ints, dim3(nblk(n, 64)), dim3(64), 0, stream, p, n);
  return hipGetLastError();
}

hipError_t launch_key(const Particles& P, const Sorted& S, const Grid& G, const StepParams& sp, DevStatus* st,
                      const VerletState& V, hipStream_t stream) {
  if (sp.n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_key, dim3(nblk(sp.n, 256)), dim3(256), 0, stream, P, S, G, sp, st, V);
  return hipGetLastError();
}

// Blocks of a gated launch (grid-stride loops): enough to fill the chip.
constexpr int kGatedBlocks = 2048;

hipError_t launch_bin(const Particles& P, const Sorted& S, const Grid& G, int n, int cx, hipStream_t stream,
                      const int* gate, const int* seq) {
  int nb = nblk(G.ncells, kScanTile);
  hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(kScanThreads), 0, stream, S.count, G.ncells, S.block_sums, gate,
                     seq);
  if (nb <= kScanFoldTiles) {
    hipLaunchKernelGGL(k_scan_down<true>, dim3(nb), dim3(kScanThreads), 0, stream, S.count, G.ncells, S.block_sums,
                       S.start, n, gate, seq);
  } else {
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(kScanThreads), 0, stream, S.block_sums, nb, gate, seq);
    hipLaunchKernelGGL(k_scan_down<false>, dim3(nb), dim3(kScanThreads), 0, stream, S.count, G.ncells, S.block_sums,
                       S.start, n, gate, seq);
  }
  // gated launches mostly find nothing to do: small grids that stride
  const int cap = gate ? kGatedBlocks : (1 << 30);
  if (n > 0) hipLaunchKernelGGL(k_scatter, dim3(std::min(nblk(n, 256), cap)), dim3(256), 0, stream, S, n, gate, seq);
  if (n > 0)
    hipLaunchKernelGGL(k_canon, dim3(std::min(nblk(n, 256), cap)), dim3(256), 0, stream, P, S, cx, n, gate, seq);
  return hipGetLastError();
}

// Verlet list build: cell keys on the list's grid (and the build positions),
// binning, then the candidates of every particle within the contact
// distance plus the skin.  Gated on the stale flag unless seq is null.
__global__ __launch_bounds__(256) void k_vkey(Particles P, Sorted S, VerletState V, int n, int cx, DevStatus* st,
                                              const int* seq, int* tcount) {
  if (tcount && blockIdx.x == 0 && threadIdx.x < kTouchLists) tcount[threadIdx.x * kItemPad] = 0;
  if (seq && st->rebuild[cx] != *seq + 1) return;  // Verlet list still valid: nothing to rebuild
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&st->n_rebuild, 1);
  const Grid& G = V.Gv;
  for (int s = blockIdx.x * blockDim.x + threadIdx.x; s < n; s += gridDim.x * blockDim.x) {
    const double x[3] = {P.x[cx][0][s], P.x[cx][1][s], P.x[cx][2][s]};
    int c[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      c[a] = min(max(ref_cell(x[a], G, a), 0), G.n[a] - 1);
      V.xb[a][s] = x[a];
    }
    const int key = (c[1] * G.n[2] + c[2]) * G.n[0] + c[0];
    S.key[s] = key;
    S.slot[s] = atomicAdd(&S.count[key], 1);
  }
}

__global__ __launch_bounds__(256) void k_vdetect(Sorted S, VerletState V, int n, NbrList L, const int* gate,
                                                 const int* seq, const DevStatus* st) {
  if (gate && *gate != *seq + 1) return;  // Verlet list still valid: nothing to rebuild
  if (st->code) return;                // an error ended the run
  const int bs = blockDim.x;
  for (int blk = xcd_tile(blockIdx.x, gridDim.x); blk * bs < n; blk += gridDim.x) {
    const int k = blk * bs + threadIdx.x;
    if (k >= n) break;
    const int s = S.order[k];
    if ((unsigned)s >= (unsigned)n) continue;
    const double* pr = S.posr + 4 * (size_t)k;
    const d3 x{pr[0], pr[1], pr[2]};
    const double r = pr[3] + V.skin;
    int c = 0;
    for_each_candidate(S, V.Gv, 0, 0, n, x, [&](int k2, int ix, int iy, int iz) {
      if (k2 == k) return;
      const double* q2 = S.posr + 4 * (size_t)k2;
      d3 xo{ix ? q2[0] + image_shift(V.Gv, 0, ix) : q2[0], iy ? q2[1] + image_shift(V.Gv, 1, iy) : q2[1],
            iz ? q2[2] + image_shift(V.Gv, 2, iz) : q2[2]};
      d3 AB = xo - x;
      double s2 = AB.x * AB.x + AB.y * AB.y + AB.z * AB.z;
      double R = r + q2[3];
      if (s2 > R * R * 1.000000000001) return;
      if (c < L.cap) L.ent[(size_t)c * n + s] = (unsigned)S.order[k2];
      ++c;
    });
    L.count[s] = c;
  }
}

hipError_t launch_verlet_build(const Particles& P, const Sorted& S, const VerletState& V, int n, int cx,
                               DevStatus* st, const NbrList& L, int* tcount, bool gated, hipStream_t stream) {
  // gated: only if the drift to these positions found the list stale
  const int* seq = gated ? &st->seq[cx] : nullptr;
  if (n == 0) return hipSuccess;
  const int nb = gated ? std::min(nblk(n, 256), kGatedBlocks) : nblk(n, 256);
  hipLaunchKernelGGL(k_vkey, dim3(nb), dim3(256), 0, stream, P, S, V, n, cx, st, seq, tcount);
  const int* gate = gated ? &st->rebuild[cx] : nullptr;
  hipError_t e = launch_bin(P, S, V.Gv, n, cx, stream, gate, seq);
  if (e != hipSuccess) return e;
  // one wave per workgroup (the candidate loops differ in length from
  // particle to particle)
  const int nb1 = gated ? std::min(nblk(n, 64), 4 * kGatedBlocks) : nblk(n, 64);
  hipLaunchKernelGGL(k_vdetect, dim3(nb1), dim3(64), 0, stream, S, V, n, L, gate, seq, st);
  return hipGetLastError();
}

int scan_blocks(int ncells) { return nblk(ncells, kScanTile); }

template <int MODE, bool MIXED>
static void launch_forces_t(const Particles& P, const Sorted& S, const Grid& G, const BoxObstacle* obs,
                            const HookeModel* models, const StepParams& sp, DevStatus* st, int* pairs,
                            const NbrList& L, const VerletState& V, const NbrList& CL, const TouchList& TL,
                            hipStream_t stream) {
  if (P.shape)
    launch_forces_shp<MODE, MIXED>(P, S, G, obs, models, sp, st, pairs, L, V, CL, stream);
  else
    launch_forces_sph<MODE, MIXED>(P, S, G, obs, models, sp, st, pairs, L, V, CL, TL, stream);
}

__global__ __launch_bounds__(256) void k_count_touched(const int* __restrict__ count, int n, int* touched) {
  int c = 0;
  for (int s = blockIdx.x * 256 + threadIdx.x; s < n; s += gridDim.x * 256) c += count[s] != 0;
  for (int d = 32; d; d >>= 1) c += __shfl_down(c, d);
  if ((threadIdx.x & 63) == 0 && c) atomicAdd(touched, c);
}
hipError_t launch_count_touched(const NbrList& CL, int n, int* touched, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipError_t e = launch_clear(touched, 1, stream);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_count_touched, dim3(std::min(nblk(n, 256), 1024)), dim3(256), 0, stream, CL.count, n, touched);
  return hipGetLastError();
}

hipError_t launch_vfilter(const Particles& P, const Sorted& S, const Grid& G, const VerletState& V, int n, int cx,
                          const NbrList& L, const NbrList& CL, const TouchList& TL, DevStatus* st, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_vfilter, dim3(nblk(n, 256)), dim3(256), 0, stream, P, S, G, V, n, cx, L, CL, TL, st);
  return hipGetLastError();
}

template <int LANES>
static void launch_detect_lanes(const Particles& P, const Sorted& S, const Grid& G, const BoxObstacle* obs,
                                const StepParams& sp, const NbrList& L, const DevStatus* st, hipStream_t stream) {
  const dim3 grid(nblk(sp.n, kDetectThreads / LANES)), block(kDetectThreads);
  if (P.shape) hipLaunchKernelGGL((k_detect<true, LANES>), grid, block, 0, stream, P, S, G, obs, sp, L, st);
  else hipLaunchKernelGGL((k_detect<false, LANES>), grid, block, 0, stream, P, S, G, obs, sp, L, st);
}

hipError_t launch_detect(const Particles& P, const Sorted& S, const Grid& G, const BoxObstacle* obs,
                         const StepParams& sp, const NbrList& L, const DevStatus* st, hipStream_t stream) {
  if (sp.n == 0) return hipSuccess;
  // lanes per particle by the number of particles, as measured (us per launch;
  // 1, 2, 4, 8 lanes): packed polyhedra 343 75, 44, 30, 22; 27,000 45, 29, 22, 20;
  // 200,000 94, 88, 83, 101; polyhedra on a loose lattice 20,000 17, 16, 14, 15;
  // 60,000 18, 18, 17, 26; 200,000 24, 35, 42, 67, and as a hopper fills with them
  // 57, 43, 49, 69, then 84, 55, 55, 74 (where the work list is another launch,
  // one lane and that launch 29, 67 and 84); packed spheres 60,000 21, 18, 17, 21,
  // 200,000 25, 26, 32, 52; gas of 27,000 23, 23, 22, 22, of 60,000 at solid
  // fraction 0.05 18, 18, 19, 22, of 1,000,000 74, 108, 151, 258.  More lanes
  // overlap the loads of few particles; once there are particles enough, every
  // lane repeats the search for the cells' runs for little.
  const bool items = P.shape != nullptr;
  if (sp.n <= 32768) launch_detect_lanes<8>(P, S, G, obs, sp, L, st, stream);
  else if (sp.n <= (items ? 65536 : 49152)) launch_detect_lanes<4>(P, S, G, obs, sp, L, st, stream);
  else if (items) launch_detect_lanes<2>(P, S, G, obs, sp, L, st, stream);
  else launch_detect_lanes<1>(P, S, G, obs, sp, L, st, stream);
  return hipGetLastError();
}

hipError_t launch_forces(int mode, bool mixed, const Particles& P, const Sorted& S, const Grid& G,
                         const BoxObstacle* obs, const HookeModel* models, const StepParams& sp, DevStatus* st,
                         int* pairs, const NbrList& L, const VerletState& V, const NbrList& CL,
                         const TouchList& TL, hipStream_t stream) {
  if (sp.n == 0) return hipSuccess;
  if (mixed) {
    if (mode == kForcesOnly) launch_forces_t<kForcesOnly, true>(P, S, G, obs, models, sp, st, pairs, L, V, CL, TL, stream);
    else if (mode == kForcesKick) launch_forces_t<kForcesKick, true>(P, S, G, obs, models, sp, st, pairs, L, V, CL, TL, stream);
    else launch_forces_t<kFused, true>(P, S, G, obs, models, sp, st, pairs, L, V, CL, TL, stream);
  } else {
    if (mode == kForcesOnly) launch_forces_t<kForcesOnly, false>(P, S, G, obs, models, sp, st, pairs, L, V, CL, TL, stream);
    else if (mode == kForcesKick) launch_forces_t<kForcesKick, false>(P, S, G, obs, models, sp, st, pairs, L, V, CL, TL, stream);
    else launch_forces_t<kFused, false>(P, S, G, obs, models, sp, st, pairs, L, V, CL, TL, stream);
  }
  return hipGetLastError();
}

}  // namespace dem
