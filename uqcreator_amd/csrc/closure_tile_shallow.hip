// closure_tile_shallow.hip -- the shallow-water instantiations of the runtime-sized
// Newton closure (closure_tile_kernel.h).
#include "closure_tile_kernel.h"

namespace uqk {

hipError_t newton_tile_shallow(int kind, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st) {
    if (kind == UQK_SHALLOW_WATER2D) return tile_kind<UQK_SHALLOW_WATER2D>(a, max_lds, num_cu, st);
    if (kind == UQK_SHALLOW_WATER2D_BARRIER) return tile_kind<UQK_SHALLOW_WATER2D_BARRIER>(a, max_lds, num_cu, st);
    return hipErrorInvalidValue;
}

}  // namespace uqk
