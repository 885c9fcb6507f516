// One-launch steps of small sphere systems, FP64 forces.
#include "dem_solo.hpp"

namespace dem {

template <int MODE>
static void launch_mode(const Particles& P, const Sorted& S, const Grid& G, const BoxObstacle* obs,
                        const HookeModel* models, const StepParams& sp, DevStatus* st, int* pairs, const NbrList& L,
                        const VerletState& V, hipStream_t stream) {
  const dim3 grid((sp.n + kSoloBodies - 1) / kSoloBodies), block(kSoloThreads);
  if (sp.mem.cap)
    hipLaunchKernelGGL((k_forces_solo<MODE, false, true>), grid, block, 0, stream, P, S, G, obs, models, sp, st, pairs, L, V);
  else
    hipLaunchKernelGGL((k_forces_solo<MODE, false, false>), grid, block, 0, stream, P, S, G, obs, models, sp, st, pairs, L, V);
}

template <>
hipError_t launch_solo_t<false>(int mode, const Particles& P, const Sorted& S, const Grid& G, const BoxObstacle* obs,
                             const HookeModel* models, const StepParams& sp, DevStatus* st, int* pairs,
                             const NbrList& L, const VerletState& V, hipStream_t stream) {
  if (mode == kForcesOnly) launch_mode<kForcesOnly>(P, S, G, obs, models, sp, st, pairs, L, V, stream);
  else if (mode == kForcesKick) launch_mode<kForcesKick>(P, S, G, obs, models, sp, st, pairs, L, V, stream);
  else launch_mode<kFused>(P, S, G, obs, models, sp, st, pairs, L, V, stream);
  return hipGetLastError();
}

}  // namespace dem
