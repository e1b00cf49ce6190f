// closure_wave_reuse.hip -- the time loop's mixed one-wavefront Newton
// closure with the reuse of the factorisation (closure_wave_kernel.h,
// PREC 2).
#include "closure_wave_kernel.h"

namespace uqk {

template <int KIND, int M, int Q>
static bool reuse_try(int kind, int m, int q, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st,
                      hipError_t* err, const LaunchShape& shape) {
    if (!wave_fits<KIND, M, Q>(kind, m, q, max_lds)) return false;
    wave_go<KIND, M, Q, 2>(a, max_lds, num_cu, st, err, shape);
    return true;
}

bool newton_wave_reuse_fits(int kind, int M, int Q, int max_lds) {
    return wave_fits<UQK_BOUNDED_BARRIER, 6, 12>(kind, M, Q, max_lds) ||
           wave_fits<UQK_EULER2D, 10, 25>(kind, M, Q, max_lds) ||
           wave_fits<UQK_SHALLOW_WATER2D, 10, 25>(kind, M, Q, max_lds) ||
           wave_fits<UQK_SHALLOW_WATER2D_BARRIER, 10, 25>(kind, M, Q, max_lds);
}

bool newton_wave_reuse_launch(int kind, int M, int Q, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st,
                              hipError_t* err, const LaunchShape& shape) {
    return reuse_try<UQK_BOUNDED_BARRIER, 6, 12>(kind, M, Q, a, max_lds, num_cu, st, err, shape) ||
           reuse_try<UQK_EULER2D, 10, 25>(kind, M, Q, a, max_lds, num_cu, st, err, shape) ||
           reuse_try<UQK_SHALLOW_WATER2D, 10, 25>(kind, M, Q, a, max_lds, num_cu, st, err, shape) ||
           reuse_try<UQK_SHALLOW_WATER2D_BARRIER, 10, 25>(kind, M, Q, a, max_lds, num_cu, st, err, shape);
}

// Floats of a cell's kept inverse for (kind, M, Q): S M rows of S M entries
// rounded up to a multiple of four.
long newton_wave_kept_floats(int S, int M) {
    const long n = (long)S * M;
    return n * ((n + 3) / 4 * 4);
}

}  // namespace uqk
