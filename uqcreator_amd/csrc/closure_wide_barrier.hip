// closure_wide_barrier.hip -- the bounded-barrier instantiations of the one-wavefront
// Newton closure for 64 duals and more (closure_wide_kernel.h).
#include "closure_wide_kernel.h"

namespace uqk {

hipError_t newton_wide_barrier(const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st, const LaunchShape& shape) {
    return wide_kind<UQK_BOUNDED_BARRIER>(a, max_lds, num_cu, st, shape);
}

hipError_t newton_wide_euler1d(const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st, const LaunchShape& shape);
hipError_t newton_wide_euler2d(const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st, const LaunchShape& shape);
hipError_t newton_wide_shallow(const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st, const LaunchShape& shape);
hipError_t newton_wide_shallow_barrier(const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st,
                                       const LaunchShape& shape);

bool newton_wide_fits(int S, int M, int Q, int max_lds) {
    return S * M <= wide_limit(S) && wide_waves(S, M, Q, max_lds) > 0;
}

long newton_wide_kept_floats(int S, int M) {
    const int nt = wide_tiles(S * M) < 6 ? 6 : wide_tiles(S * M);
    return 256l * (nt * (nt + 1) / 2);
}

hipError_t newton_wide_launch(int kind, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st,
                              const LaunchShape& shape) {
    switch (kind) {
        case UQK_BOUNDED_BARRIER: return newton_wide_barrier(a, max_lds, num_cu, st, shape);
        case UQK_EULER1D: return newton_wide_euler1d(a, max_lds, num_cu, st, shape);
        case UQK_EULER2D: return newton_wide_euler2d(a, max_lds, num_cu, st, shape);
        case UQK_SHALLOW_WATER2D: return newton_wide_shallow(a, max_lds, num_cu, st, shape);
        case UQK_SHALLOW_WATER2D_BARRIER: return newton_wide_shallow_barrier(a, max_lds, num_cu, st, shape);
    }
    return hipErrorInvalidValue;
}

}  // namespace uqk
