// One-launch steps of small sphere systems, FP64 forces.
#include "dem_solo.hpp"

namespace dem {

template hipError_t launch_solo_t<false>(int, const Particles&, const Sorted&, const Grid&, const BoxObstacle*, const HookeModel*,
    const StepParams&, DevStatus*, int*, const NbrList&, const VerletState&, hipStream_t);

}  // namespace dem
