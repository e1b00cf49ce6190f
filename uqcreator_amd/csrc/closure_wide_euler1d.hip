// closure_wide_euler1d.hip -- the Euler 1D instantiations of the one-wavefront
// Newton closure for 64 duals and more (closure_wide_kernel.h).
#include "closure_wide_kernel.h"

namespace uqk {

hipError_t newton_wide_euler1d(const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st, const LaunchShape& shape) {
    return wide_kind<UQK_EULER1D>(a, max_lds, num_cu, st, shape);
}

}  // namespace uqk
