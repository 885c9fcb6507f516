// The step of a small system of spheres with a Verlet list in one launch:
// rebuild of the list when it is stale, contacts, forces, integration (shared
// by the per-precision translation units dem_solo*.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dem_forces.hpp"
#include "dem_launch.hpp"

namespace dem {

// A step of a small system is waiting: launches (seven empty ones besides two
// with work), and in the force sweep a lane that walks its contacts one after
// the other, each a chain of gathers and some forty correctly rounded
// divisions and roots.  Here kSoloThreads / kSoloBodies lanes share a
// particle: the listed neighbours of a workgroup's particles are spread over
// its lanes, one per lane, the force and torque of each contact left in LDS and
// summed by the particle's thread in the list's order -- the sum of the general
// sweep, but for a law with a rolling moment, which joins its contact's torque
// before that sum and not after it (one rounding of the torque per contact).
// Pairs first, then obstacles, as there, each kind in waves of its own.
// Bound by the latency of one contact and of the phases' barriers.  Per step,
// general launches -> this one: bed of 1,000 41 -> 18.8 us, of 48,611 (mixed)
// 39 -> 20, 5,003 with contact memory 72 -> 29, gas of 27,000 37 -> 18, of 64,000
// 37 -> 25.  Above, gases are as fast or faster by the general launches, with
// more waves on the streaming part (110,000 43.7 against 47.8 us, 200,000 49
// against 73), beds from somewhere above 100,000 (100,000 71 against 56, 200,000
// 80 against 93); the rule stands at grains_gpu_system::kSoloMax.
constexpr int kSoloThreads = 256;
constexpr int kSoloBodies = 64;

// ---------------------------------------------------------------------------
// Verlet list rebuild inside the sweep.  The work of its phases (cell keys,
// cell counts to starts, places, ranks, neighbours) is cut into pieces that the
// workgroups take in order from one counter; a piece of a phase first waits
// until every piece of the phase before is done.  A workgroup only waits for
// pieces taken earlier, whose workgroups are running and wait for still earlier
// ones, so the first piece not yet done never waits and all end, whatever share
// of the launch is resident.
// A piece is published by one wave for the workgroup, and its predecessors'
// are taken up by one wave, once per phase: every agent-scope fence writes back
// or invalidates the XCD's L2, and with a fence per wave and piece they were
// what a rebuild waited for (a step of a gas of 64,000 that rebuilds every
// fourth or fifth time 87 us, 70 with one).  The stores of all waves have
// reached the L2 (s_waitcnt) before the barrier, so the one write-back covers
// them; the count is raised when it has ended, which is waited for explicitly:
// with no store
// of this wave outstanding the compiler leaves that wait out.
__device__ __forceinline__ void drain() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void wait_pieces(int* done, int count) {
  if (threadIdx.x == 0) {
    // (hundreds of waiting workgroups that ask often hold up the counts)
    while (__hip_atomic_load(done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < count) {
      if (gridDim.x > 256) __builtin_amdgcn_s_sleep(16);
      else __builtin_amdgcn_s_sleep(2);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    drain();
  }
  __syncthreads();
}
__device__ __forceinline__ void piece_done(int* done) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  drain();
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    drain();
    __hip_atomic_fetch_add(done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// inclusive sum over the workgroup (kSoloThreads lanes); total of all lanes
__device__ __forceinline__ int block_sum_scan(int v, int* lds, int& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int incl = v;
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(incl, d);
    if (lane >= d) incl += u;
  }
  __syncthreads();
  if (lane == 63) lds[w] = incl;
  __syncthreads();
  total = 0;
  for (int k = 0; k < kSoloThreads / 64; ++k) {
    if (k < w) incl += lds[k];
    total += lds[k];
  }
  return incl;
}

// Small pieces fill the chip, but each is published with a write-back of its
// XCD's L2: about 250 pieces of the neighbour phase at most (us per step that
// rebuilds every fourth or fifth time, of a gas of 8,000, 27,000 and 64,000: 25,
// 37 and 59; four times as many 25, 42 and 79; 1,024 particles to every piece of
// the other phases and 128 to those of this one 33, 47 and 70).
constexpr int kPieceStep = 16384;              // particles per round of a piece's threads
constexpr int kPieceCells = 8 * kSoloThreads;  // phases over cells
constexpr int kSearchLanes = 4;                // lanes per particle of the neighbour phase

__device__ __forceinline__ void solo_rebuild(const Particles& P, const Sorted& S, const VerletState& V, const NbrList& L,
                                          int n, int cx, DevStatus* st) {
  __shared__ int ticket, lds[4];
  RebuildSync* const rs = V.sync + cx;
  const Grid& G = V.Gv;
  const int tid = threadIdx.x;
  const int rounds = 1 + n / kPieceStep, bodies = rounds * kSoloThreads, search = bodies / kSearchLanes;
  const int nb = (n + bodies - 1) / bodies, nc = (G.ncells + kPieceCells - 1) / kPieceCells;
  const int count[6] = {nb, nc, nc, nb, nb, (n + search - 1) / search};
  int seen = 0;  // pieces of this phase were waited for
  for (;;) {
    __syncthreads();
    if (tid == 0) ticket = __hip_atomic_fetch_add(&rs->ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    int i = ticket, phase = 0;
    while (phase < 6 && i >= count[phase]) i -= count[phase++];
    if (phase == 6) break;
    if (phase > seen) {
      wait_pieces(&rs->done[phase - 1], count[phase - 1]);
      seen = phase;
    }
    if (phase == 0) {
      // cell keys on the list's grid, build positions
      if (i == 0 && tid == 0) atomicAdd(&st->n_rebuild, 1);
      for (int s = i * bodies + tid; s < min((i + 1) * bodies, n); s += kSoloThreads) {
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
    } else if (phase == 1 || phase == 2) {
      // sums of the cells' counts, then their starts
      int before = 0, sums;
      if (phase == 2) {
        int part = 0;
        for (int b = tid; b < i; b += kSoloThreads) part += S.block_sums[b];
        block_sum_scan(part, lds, before);
      }
      const int c0 = i * kPieceCells + tid * 8;
      int v[8], sum = 0;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        v[k] = c0 + k < G.ncells ? S.count[c0 + k] : 0;
        sum += v[k];
      }
      int run = before + block_sum_scan(sum, lds, sums) - sum;
      if (phase == 1) {
        if (tid == 0) S.block_sums[i] = sums;
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          if (c0 + k < G.ncells) {
            S.start[c0 + k] = run;
            S.count[c0 + k] = 0;
          }
          run += v[k];
        }
        if (i == 0 && tid == 0) S.start[G.ncells] = n;
      }
    } else if (phase == 3) {
      for (int s = i * bodies + tid; s < min((i + 1) * bodies, n); s += kSoloThreads) {
        const int dst = S.start[S.key[s]] + S.slot[s];
        if ((unsigned)dst < (unsigned)n) S.tmp_order[dst] = s;
      }
    } else if (phase == 4) {
      for (int j = i * bodies + tid; j < min((i + 1) * bodies, n); j += kSoloThreads)
        rank_particle(P, S, j, cx, n);
    } else {
      // neighbours within the contact distance plus the skin, kSearchLanes
      // candidates at a time in the order of the cells
      const int lane = tid & (kSearchLanes - 1), gshift = tid & 63 & ~(kSearchLanes - 1);
      for (int k = i * search + tid / kSearchLanes; k < min((i + 1) * search, n);
           k += kSoloThreads / kSearchLanes) {
        const int s = S.order[k];
        if ((unsigned)s >= (unsigned)n) continue;
        const double* pr = S.posr + 4 * (size_t)k;
        const d3 x{pr[0], pr[1], pr[2]};
        const double r = pr[3] + V.skin;
        int c = 0;
        for_each_run(S, G, 0, 0, n, x, [&](int b, int e, int ix, int iy, int iz) {
          for (int k0 = b; k0 < e; k0 += kSearchLanes) {
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
            const unsigned hits = (unsigned)(__ballot(hit) >> gshift) & ((1u << kSearchLanes) - 1u);
            const int j = c + __popc(hits & ((1u << lane) - 1u));
            if (hit && j < L.cap) L.ent[(size_t)j * n + s] = (unsigned)S.order[k2];
            c += __popc(hits);
          }
        });
        if (lane == 0) L.count[s] = c;
      }
    }
    piece_done(&rs->done[phase]);
  }
  wait_pieces(&rs->done[5], count[5]);
}

// ---------------------------------------------------------------------------
// MEM: contact models with memory.  A particle's entries are numbered by its
// earlier contacts whose material pair has memory (a mask per particle): pairs
// of a plain Hooke law, which write none, may stand between them.
template <bool MIXED, bool MEM>
using TermT = std::conditional_t<MIXED && !MEM, float, double>;

template <int MODE, bool MIXED, bool MEM>
__global__ __launch_bounds__(kSoloThreads) __attribute__((amdgpu_waves_per_eu(2))) void k_forces_solo(
    Particles P, Sorted S, Grid G, const BoxObstacle* __restrict__ obs, const HookeModel* __restrict__ models,
    StepParams sp, DevStatus* st, int* pairs, NbrList L, VerletState VS) {
  constexpr int T = kSoloThreads, B = kSoloBodies;
  static_assert(B == 64, "the offsets are scanned by one wave");
  using FV = ForceVisitor<MIXED, MEM, false>;
  using Term = TermT<MIXED, MEM>;
  __shared__ double self[11][B];
  __shared__ Term term[6][T];
  __shared__ Term termc[MIXED && MEM ? 6 : 1][MIXED && MEM ? T : 1];  // 32-bit sums beside the 64-bit ones
  __shared__ unsigned short owner[T], index[T];
  __shared__ int total_of[2];
  __shared__ unsigned long long touch[MEM ? B : 1];
  __shared__ int rank0[MEM ? B : 1];  // memory entries of the particle's earlier contacts
  const int tid = threadIdx.x;
  const int t0 = xcd_tile(blockIdx.x, gridDim.x) * B;
  const int cx = sp.cur & 1, cv = (sp.cur >> 1) & 1;
  // after an error (which ends the run) the rest of a batch of steps neither
  // rebuilds nor searches, so that it costs little whatever the state has become
  const bool stop = st->stop[cx] != 0;
  if (!stop && VS.stamp == 1 && st->rebuild[cx] == st->seq[cx] + 1) solo_rebuild(P, S, VS, L, sp.n, cx, st);
  if (MODE == kFused) number_next(sp, st, VS);
  const bool mine = tid < B && t0 + tid < sp.n;
  const int s = t0 + tid;
  int c = 0, cw = 0;
  bool over = false;
  unsigned long long walls = 0ull;
  d3 F{0., 0., 0.}, Tq{0., 0., 0.};
  f3 Fc{0.f, 0.f, 0.f}, Tc{0.f, 0.f, 0.f};
  if (mine) {
    const d3 x = ld3(P.x[cx], s), v = ld3(P.v[cv], s), w = ld3(P.w[cv], s);
    const double r = P.rad[s], wf = P.wfac[s];
    const double a[11] = {x.x, x.y, x.z, v.x, v.y, v.z, w.x, w.y, w.z, r, P.mass[s]};
#pragma unroll
    for (int k = 0; k < 11; ++k) self[k][tid] = a[k];
    // InitializeForce: torsor = weight at the centre (Particle.cpp:1408-1415)
    F = d3{sp.g[0] * wf, sp.g[1] * wf, sp.g[2] * wf};
    c = stop ? 0 : L.count[s];
    over = c > L.cap;
    if (over) c = 0;
    const int nobs = stop ? 0 : sp.nobs;
    for (int o = 0; o < nobs; ++o)
      if (near_obstacle(obs[o], x, r)) walls |= 1ull << o;
    cw = over ? 0 : __popcll(walls);
  }
  if (MEM && tid < B) rank0[tid] = 0;
  // a particle of the block as its contacts see it
  auto body = [&](int p) {
    Self me;
    me.x = d3{self[0][p], self[1][p], self[2][p]};
    me.v = d3{self[3][p], self[4][p], self[5][p]};
    me.w = d3{self[6][p], self[7][p], self[8][p]};
    me.r = self[9][p];
    me.m = self[10][p];
    me.c = P.crust[t0 + p];
    me.req = P.req[t0 + p];
    me.mat = P.mat[t0 + p];
    me.id = P.id[t0 + p];
    return me;
  };
  auto pair_of = [&](const Self& me, int s2i, d3& xo, double& ro, d3& Pc, d3& ov, double& d) {
    const d3 x2{P.x[cx][0][s2i], P.x[cx][1][s2i], P.x[cx][2][s2i]};
    ro = P.rad[s2i];
    xo = nearest_image(G, x2, me.x);
    const d3 AB = xo - me.x;
    const double s2 = AB.x * AB.x + AB.y * AB.y + AB.z * AB.z, R = me.r + ro;
    if (s2 > R * R * 1.000000000001) return false;
    const int id2 = P.id[s2i];
    return sphere_features(st, me, P.crust[s2i], IdAt{&id2}, xo, ro, AB, sqrt(s2), Pc, ov, d) && d < 0.;
  };
  // exclusive offsets of n items per particle over the block; returns the total
  auto offsets = [&](int n, int which, int& off) {
    if (tid < 64) {
      int incl = n;
      for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(incl, d);
        if (tid >= d) incl += u;
      }
      off = incl - n;
      if (tid == 63) total_of[which] = incl;
    }
    __syncthreads();
    return total_of[which];
  };
  // the items of one kind: window after window of T, one per lane; features
  // also says whether the pair's law has memory
  auto sweep = [&](int n, int which, auto&& entry, auto&& features, auto&& force) {
    int off = 0;
    const int total = offsets(n, which, off);
    for (int base = 0; base < total; base += T) {
      for (int i = max(0, base - off); i < n && off + i < base + T; ++i) {
        owner[off + i - base] = (unsigned short)tid;
        index[off + i - base] = (unsigned short)entry(i);
      }
      if (MEM && tid < B) touch[tid] = 0ull;
      __syncthreads();
      const bool item = base + tid < total;
      const int p = item ? owner[tid] : 0, e = item ? index[tid] : 0;
      Self me;
      d3 Pc, ov, xo{0., 0., 0.};
      double d = 0., ro = 0.;
      int partner = 0;
      bool live = false, memory = false;
      if (item) {
        me = body(p);
        live = features(me, p, e, partner, memory, xo, ro, Pc, ov, d);
      }
      FV vis{P, S, obs, models, sp, st, pairs, cv, me, d3{0., 0., 0.}, d3{0., 0., 0.}, f3{0.f, 0.f, 0.f},
             f3{0.f, 0.f, 0.f}};
      if (MEM) {
        // (the window holds items of rising index per particle: bit e)
        if (live && memory) atomicOr(&touch[p], 1ull << (e & 63));
        __syncthreads();
        vis.s = t0 + p;
        if (live) vis.nmem = rank0[p] + __popcll(touch[p] & ((1ull << (e & 63)) - 1ull));
      }
      if (live) force(vis, partner, xo, ro, Pc, ov, d);
      if (MIXED && !MEM) {
        const float a[6] = {vis.Fc.x, vis.Fc.y, vis.Fc.z, vis.Tc.x, vis.Tc.y, vis.Tc.z};
#pragma unroll
        for (int k = 0; k < 6; ++k) term[k][tid] = (Term)a[k];
      } else {
        const double a[6] = {vis.F.x, vis.F.y, vis.F.z, vis.T.x, vis.T.y, vis.T.z};
#pragma unroll
        for (int k = 0; k < 6; ++k) term[k][tid] = (Term)a[k];
        if (MIXED && MEM) {
          const float b[6] = {vis.Fc.x, vis.Fc.y, vis.Fc.z, vis.Tc.x, vis.Tc.y, vis.Tc.z};
#pragma unroll
          for (int k = 0; k < 6; ++k) termc[k][tid] = (Term)b[k];
        }
      }
      __syncthreads();
      if (tid < B) {
        for (int i = max(0, base - off); i < n && off + i < base + T; ++i) {
          const int j = off + i - base;
          if (MIXED && !MEM) {
            Fc += f3{(float)term[0][j], (float)term[1][j], (float)term[2][j]};
            Tc += f3{(float)term[3][j], (float)term[4][j], (float)term[5][j]};
          } else {
            F += d3{(double)term[0][j], (double)term[1][j], (double)term[2][j]};
            Tq += d3{(double)term[3][j], (double)term[4][j], (double)term[5][j]};
            if (MIXED && MEM) {
              Fc += f3{(float)termc[0][j], (float)termc[1][j], (float)termc[2][j]};
              Tc += f3{(float)termc[3][j], (float)termc[4][j], (float)termc[5][j]};
            }
          }
        }
        if (MEM) rank0[tid] += __popcll(touch[tid]);
      }
      // the window's arrays are written again
      if (base + T < total) __syncthreads();
    }
    return total;
  };
  sweep(
      c, 0, [](int i) { return i; },
      [&](const Self& me, int p, int e, int& partner, bool& memory, d3& xo, double& ro, d3& Pc, d3& ov, double& d) {
        const unsigned s2i = L.ent[(size_t)e * L.n + t0 + p];
        partner = (int)s2i;
        if (s2i >= (unsigned)sp.n) return false;
        if (MEM) memory = models[me.mat * kMaxMaterials + P.mat[s2i]].memory != 0;
        return pair_of(me, (int)s2i, xo, ro, Pc, ov, d);
      },
      [&](FV& vis, int s2i, d3 xo, double ro, d3 Pc, d3 ov, double d) {
        const int id2 = P.id[s2i];
        vis.pair(-1, s2i, IdAt{&id2}, xo, ro, Pc, ov, d);
      });
  if (sp.nobs) {
    __syncthreads();
    unsigned long long left = over ? 0ull : walls;
    sweep(
        cw, 1,
        [&](int) {
          const int o = __builtin_ctzll(left);
          left &= left - 1ull;
          return o;
        },
        [&](const Self& me, int, int e, int& partner, bool& memory, d3&, double&, d3& Pc, d3& ov, double& d) {
          partner = e;
          if (MEM) memory = models[me.mat * kMaxMaterials + obs[e].mat].memory != 0;
          return wall_features(obs[e], st, me, Pc, ov, d) && d < 0.;
        },
        [&](FV& vis, int o, d3, double, d3 Pc, d3 ov, double d) { vis.wall(o, Pc, ov, d); });
  }
  if (!mine) return;
  if (over) {
    // more neighbours than the list holds: the particle's thread searches the
    // cells around its build position
    const Self me = body(tid);
    FV vis{P, S, obs, models, sp, st, pairs, cv, me, F, Tq, f3{0.f, 0.f, 0.f}, f3{0.f, 0.f, 0.f}};
    vis.s = s;
    auto one = [&](int s2i) {
      d3 xo, Pc, ov;
      double ro, d = 0.;
      if (pair_of(me, s2i, xo, ro, Pc, ov, d)) vis.pair(-1, s2i, IdAt{P.id + s2i}, xo, ro, Pc, ov, d);
    };
    const d3 xb{VS.xb[0][s], VS.xb[1][s], VS.xb[2][s]};
    for_each_candidate(S, VS.Gv, 0, 0, sp.n, xb, [&](int k2, int, int, int) {
      const int s2i = S.order[k2];
      if (s2i != s && (unsigned)s2i < (unsigned)sp.n) one(s2i);
    });
    for (int o = 0; o < sp.nobs; ++o) {
      d3 Pc, ov;
      double d = 0.;
      if ((walls >> o & 1ull) && wall_features(obs[o], st, me, Pc, ov, d) && d < 0.) vis.wall(o, Pc, ov, d);
    }
    F = vis.F;
    Tq = vis.T;
    Fc = vis.Fc;
    Tc = vis.Tc;
    if (MEM) rank0[tid] = vis.nmem;
  }
  if (MIXED) {
    F += d3{(double)Fc.x, (double)Fc.y, (double)Fc.z};
    Tq += d3{(double)Tc.x, (double)Tc.y, (double)Tc.z};
  }
  if (MEM && sp.mem.cap) {
    // this evaluation's contact memory of the particle (every particle, so
    // that entries of contacts that ended are dropped)
    sp.mem.n[sp.mem.cur ^ 1][s] = min(rank0[tid], sp.mem.cap);
    if (rank0[tid] > sp.mem.cap) raise_error(st, kMemoryOverflow, P.id[s], rank0[tid]);
  }
  // forces of the fluid (AppPRSHydroFT::ComputeForces, AppPRSHydroFT.cpp:
  // 27-44): an application after the contacts, the force at the centre
  if (sp.hyd) {
    const size_t n = (size_t)sp.n;
    F += d3{sp.hyd[s], sp.hyd[n + s], sp.hyd[2 * n + s]};
    Tq += d3{sp.hyd[3 * n + s], sp.hyd[4 * n + s], sp.hyd[5 * n + s]};
  }
  if (!(MODE == kFused && sp.scheme == kLeapFrog)) {
    st3(P.F, s, F);
    st3(P.T, s, Tq);
  }
  if (MODE == kForcesOnly) return;
  Kin kin;
  kin.x = d3{self[0][tid], self[1][tid], self[2][tid]};
  kin.v = d3{self[3][tid], self[4][tid], self[5][tid]};
  kin.w = d3{self[6][tid], self[7][tid], self[8][tid]};
  kin.wb = ld3(P.wb, s);
  kin.q = quat{d3{P.q[0][s], P.q[1][s], P.q[2][s]}, P.q[3][s]};
  sphere_tail<MODE>(P, S, G, sp, st, VS, s, cx, cv, kin, self[10][tid], P.crust[s], P.cfac[s], P.inertia[s], F, Tq);
}

template <int MODE, bool MIXED>
static void launch_solo_mode(const Particles& P, const Sorted& S, const Grid& G, const BoxObstacle* obs,
                             const HookeModel* models, const StepParams& sp, DevStatus* st, int* pairs,
                             const NbrList& L, const VerletState& V, hipStream_t stream) {
  const dim3 grid((sp.n + kSoloBodies - 1) / kSoloBodies), block(kSoloThreads);
  if (sp.mem.cap)
    hipLaunchKernelGGL((k_forces_solo<MODE, MIXED, true>), grid, block, 0, stream, P, S, G, obs, models, sp, st, pairs, L, V);
  else
    hipLaunchKernelGGL((k_forces_solo<MODE, MIXED, false>), grid, block, 0, stream, P, S, G, obs, models, sp, st, pairs, L, V);
}

// (instantiated once per precision, each in a translation unit of its own)
template <bool MIXED>
hipError_t launch_solo_t(int mode, const Particles& P, const Sorted& S, const Grid& G, const BoxObstacle* obs,
                         const HookeModel* models, const StepParams& sp, DevStatus* st, int* pairs, const NbrList& L,
                         const VerletState& V, hipStream_t stream) {
  if (mode == kForcesOnly) launch_solo_mode<kForcesOnly, MIXED>(P, S, G, obs, models, sp, st, pairs, L, V, stream);
  else if (mode == kForcesKick) launch_solo_mode<kForcesKick, MIXED>(P, S, G, obs, models, sp, st, pairs, L, V, stream);
  else launch_solo_mode<kFused, MIXED>(P, S, G, obs, models, sp, st, pairs, L, V, stream);
  return hipGetLastError();
}

}  // namespace dem
