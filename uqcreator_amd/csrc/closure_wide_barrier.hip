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

// The kernel is taken where it is the faster one (8,192 cells, one closure in
// FP64, against the workgroup kernel as it is resident): with four wavefronts
// in LDS beside the tables 0.23..0.34 of its time, with three 0.25..0.46, with
// two 0.38..0.71; with one, which leaves three SIMDs idle, 1.00..1.42 where two
// workgroups are resident (n = 105: 9.8 ms against 7.9 at 216 points), and
// 0.77..0.84 where one is (n = 112, 124).  With one state a cell is one long
// chain for its wavefront (every basis pair, and one product in four used), so
// as many cells as workgroups are resident go to the workgroup kernel (n = 64,
// 66 points: 64 cells 0.45 ms against 0.32, 512 cells 0.47 against 0.38), more
// of them here (1,024 cells 0.48 against 0.68).
bool newton_wide_takes(int S, int M, int Q, int max_lds, int num_cu, long ncell) {
    const int waves = S * M <= wide_limit(S) ? wide_waves(S, M, Q, max_lds) : 0;
    if (waves == 0 || !newton_block_fits(S, M, Q, max_lds)) return waves > 0;
    const int resident = 2 * newton_block_lds(S, M, Q) <= (size_t)max_lds ? 2 : 1;
    if (waves == 1 && resident == 2) return false;
    return S > 1 || ncell > (long)resident * num_cu;
}

long newton_wide_kept_floats(int S, int M) { return wide_kept(S * M); }

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
