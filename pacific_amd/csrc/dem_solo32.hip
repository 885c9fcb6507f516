// One-launch steps of small sphere systems, mixed-precision forces.
#include "dem_solo.hpp"

namespace dem {

template hipError_t launch_solo_t<true>(int, const Particles&, const Sorted&, const Grid&, const BoxObstacle*, const HookeModel*,
    const StepParams&, DevStatus*, int*, const NbrList&, const VerletState&, hipStream_t);
extern template hipError_t launch_solo_t<false>(int, const Particles&, const Sorted&, const Grid&, const BoxObstacle*, const HookeModel*,
    const StepParams&, DevStatus*, int*, const NbrList&, const VerletState&, hipStream_t);

hipError_t launch_forces_solo(int mode, bool mixed, const Particles& P, const Sorted& S, const Grid& G,
                              const BoxObstacle* obs, const HookeModel* models, const StepParams& sp, DevStatus* st,
                              int* pairs, const NbrList& L, const VerletState& V, hipStream_t stream) {
  if (sp.n == 0) return hipSuccess;
  return mixed ? launch_solo_t<true>(mode, P, S, G, obs, models, sp, st, pairs, L, V, stream)
               : launch_solo_t<false>(mode, P, S, G, obs, models, sp, st, pairs, L, V, stream);
}

}  // namespace dem
