// closure_tile_euler2d.hip -- the Euler 2D instantiations of the runtime-sized
// Newton closure (closure_tile_kernel.h).
#include "closure_tile_kernel.h"

namespace uqk {

hipError_t newton_tile_euler2d(int kind, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st) {
    if (kind == UQK_EULER2D) return tile_kind<UQK_EULER2D>(a, max_lds, num_cu, st);
    return hipErrorInvalidValue;
}

}  // namespace uqk
