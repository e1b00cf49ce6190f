// closure_tile_euler1d.hip -- the Euler 1D instantiations of the runtime-sized
// Newton closure (closure_tile_kernel.h).
#include "closure_tile_kernel.h"

namespace uqk {

hipError_t newton_tile_euler1d(int kind, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st) {
    if (kind == UQK_EULER1D) return tile_kind<UQK_EULER1D>(a, max_lds, num_cu, st);
    return hipErrorInvalidValue;
}

}  // namespace uqk
