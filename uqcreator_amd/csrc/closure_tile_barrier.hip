// closure_tile_barrier.hip -- the bounded barrier instantiations of the runtime-sized
// Newton closure (closure_tile_kernel.h).
#include "closure_tile_kernel.h"

namespace uqk {

hipError_t newton_tile_barrier(int kind, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st) {
    if (kind == UQK_BOUNDED_BARRIER) return tile_kind<UQK_BOUNDED_BARRIER>(a, max_lds, num_cu, st);
    return hipErrorInvalidValue;
}

hipError_t newton_tile_euler1d(int kind, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st);
hipError_t newton_tile_euler2d(int kind, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st);
hipError_t newton_tile_shallow(int kind, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st);

bool newton_tile_fits(int S, int M, int Q, int max_lds) {
    const TileLds at(S, M, Q);
    return S * M < 64 && sizeof(double) * ((size_t)at.tables + at.wave) <= (size_t)max_lds;
}

hipError_t newton_tile_launch(int kind, const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st) {
    switch (kind) {
        case UQK_BOUNDED_BARRIER: return newton_tile_barrier(kind, a, max_lds, num_cu, st);
        case UQK_EULER1D: return newton_tile_euler1d(kind, a, max_lds, num_cu, st);
        case UQK_EULER2D: return newton_tile_euler2d(kind, a, max_lds, num_cu, st);
    }
    return newton_tile_shallow(kind, a, max_lds, num_cu, st);
}

}  // namespace uqk
