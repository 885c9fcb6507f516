// Host entry points of the DEM kernels (dem_kernels.hip)
#pragma once
#include <hip/hip_runtime.h>

#include "dem_types.hpp"

namespace dem {

enum ForceMode { kModeForcesOnly = 0, kModeForcesKick = 1, kModeFused = 2 };

// first half kick + drift (or a full Move of the explicit schemes) in place,
// then cell key and arrival slot; number: the number of the positions written
// (DevStatus::seq)
hipError_t launch_move(const Particles& P, const Sorted& S, const Grid& G, const StepParams& sp, DevStatus* st,
                       double dtv, double dtx, const VerletState& V, int number, hipStream_t stream);
// cell key and arrival slot of the current positions (no motion)
hipError_t launch_key(const Particles& P, const Sorted& S, const Grid& G, const StepParams& sp, DevStatus* st,
                      const VerletState& V, hipStream_t stream);
// counts -> start, scatter, per-cell ordering; cx = position buffer to gather;
// with gate, only when *gate == *seq + 1
hipError_t launch_bin(const Particles& P, const Sorted& S, const Grid& G, int n, int cx, hipStream_t stream,
                      const int* gate = nullptr, const int* seq = nullptr);
// Verlet list build (keys on its grid, binning, candidates) from position
// buffer cx; gated: only if the drift that wrote it found the list stale
hipError_t launch_verlet_build(const Particles& P, const Sorted& S, const VerletState& V, int n, int cx,
                               DevStatus* st, const NbrList& L, int* tcount, bool gated, hipStream_t stream);
int scan_blocks(int ncells);
// zero n ints with a kernel (safe inside captured graphs, unlike hipMemsetAsync)
hipError_t launch_clear(int* p, int n, hipStream_t stream);
// contacts of this step from the Verlet list L into CL, and the particles that
// have one into TL (if kept)
hipError_t launch_vfilter(const Particles& P, const Sorted& S, const Grid& G, const VerletState& V, int n, int cx,
                          const NbrList& L, const NbrList& CL, const TouchList& TL, DevStatus* st, hipStream_t stream);
// folds the per-block contact statistics of the last force launch over n
// particles into the running totals (6 doubles), at the given time
hipError_t launch_stats_fold(const double* part, int n, double* tot, double time, hipStream_t stream);
// particles with a contact in CL (of n) into *touched
hipError_t launch_count_touched(const NbrList& CL, int n, int* touched, hipStream_t stream);
// neighbour candidates of every sorted particle into L, and, for a system
// with non-spherical bodies, the narrow phase's work list into sp.cf
hipError_t launch_detect(const Particles& P, const Sorted& S, const Grid& G, const BoxObstacle* obs,
                         const StepParams& sp, const NbrList& L, const DevStatus* st, hipStream_t stream);
// threads of a workgroup of the contact search, and bodies at most (its work
// list is sized for any number of lanes per body)
constexpr int kDetectThreads = 256;
// narrow phase of a system with non-spherical bodies: the contacts of every
// sorted particle (candidates of L, or its 27 cells when L.count is null)
// into sp.cf, and the contact statistics when sp.stats is set
hipError_t launch_narrow(const Particles& P, const Sorted& S, const Grid& G, const BoxObstacle* obs,
                         const StepParams& sp, DevStatus* st, const NbrList& L, hipStream_t stream);
// force sweep of a small system of spheres with a Verlet list, which it
// rebuilds itself when it is stale (k_forces_solo)
hipError_t launch_forces_solo(int mode, bool mixed, const Particles& P, const Sorted& S, const Grid& G,
                              const BoxObstacle* obs, const HookeModel* models, const StepParams& sp, DevStatus* st,
                              int* pairs, const NbrList& L, const VerletState& V, hipStream_t stream);
// force sweep over the candidates of L (L.count == nullptr: 27-cell sweep)
hipError_t launch_forces(int mode, bool mixed, const Particles& P, const Sorted& S, const Grid& G,
                         const BoxObstacle* obs, const HookeModel* models, const StepParams& sp, DevStatus* st,
                         int* pairs, const NbrList& L, const VerletState& V, const NbrList& CL,
                         const TouchList& TL, hipStream_t stream);

}  // namespace dem
