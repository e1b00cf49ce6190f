// cell_queue.h -- how the wavefronts of a closure launch share the cells, and
// how they add up their counts.
//
// Cells differ in cost (Newton steps), but most of them can be dealt out
// beforehand: three quarters of a launch's cells go to its wavefronts in
// rounds (position w of round t is wavefront w's), which spreads clusters of
// costly cells over all of them, and only the last quarter is taken from a
// counter, one cell at a time.  An atomic on one address costs about 12 ns
// here whatever its scope's load, all atomics on it in sequence: 2,000
// wavefronts that each ask once and add five counts at the end took 40 us for
// 400 cells.  So the counter is split over kCounterLines cache lines (the
// wavefronts of a group share one, and the tail's cells are dealt to the
// groups in turn), counts are added per workgroup to the group's line, and a
// launch with no more cells than wavefronts takes no ticket at all.
#pragma once

#include <hip/hip_runtime.h>

#include "uqk_internal.h"

namespace uqk {

// The cells of one wavefront.  Use: first() gives its first position; at the
// start of a cell ask() sends for the next one, resolve() -- some hundred
// cycles later -- turns the ticket into a cell (a load from the list), take()
// -- when the cell ends -- returns it; none of the three waits for memory if
// that much time has passed.
struct CellQueue {
    long total, workers, pos;
    long rounds;       // rounds dealt out beforehand
    long round = 0;
    const int* list;   // position -> cell (null: the cell is the position)
    unsigned long long* ticket_at;
    int group, groups;  // of workgroups, kCounterLines where there are as many
    unsigned ticket = 0;
    int cell = -1;

    __device__ __forceinline__ CellQueue(long worker, long nworkers, long ncells, const int* cells,
                                         unsigned long long* counters)
        : total(ncells), workers(nworkers), pos(worker), list(cells),
          groups(gridDim.x < kCounterLines ? gridDim.x : kCounterLines) {
        group = blockIdx.x % groups;
        ticket_at = counters + group * kCounterLine;
        const long all = (ncells + nworkers - 1) / nworkers;
        rounds = all <= 1 ? 1 : (3 * (ncells / nworkers)) / 4;
        if (rounds < 1) rounds = 1;
    }
    __device__ __forceinline__ void ask() {
        ++round;
        if (round >= rounds && (threadIdx.x & 63) == 0 && rounds * workers < total)
            ticket = (unsigned)atomicAdd(ticket_at, 1ull);
    }
    __device__ __forceinline__ void resolve() {
        long p = pos + round * workers;
        if (round >= rounds)
            p = rounds * workers < total
                    ? rounds * workers + (long)(unsigned)__builtin_amdgcn_readfirstlane(ticket) * groups + group
                    : total;
        cell = p < total ? (list ? list[p] : (int)p) : -1;
    }
    __device__ __forceinline__ long take() const { return (long)__builtin_amdgcn_readfirstlane(cell); }
    __device__ __forceinline__ long first() {
        cell = pos < total ? (list ? list[pos] : (int)pos) : -1;
        return take();
    }
};

// Adds a workgroup's counts (per wavefront: v[1..6] of the counters' order)
// and its smallest ComputeDt to the launch's.  scratch: 8 doubles per
// wavefront of LDS that no wavefront uses any more.  Every thread calls it.
__device__ __forceinline__ void add_counts(const unsigned long long (&v)[7], double dt, double* scratch,
                                           unsigned long long* counters, unsigned long long* dt_min) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    unsigned long long* s = reinterpret_cast<unsigned long long*>(scratch);
    __syncthreads();
    if (lane == 0) {
#pragma unroll
        for (int i = 1; i < 7; ++i) s[wave * 8 + i] = v[i];
        scratch[wave * 8] = dt;
    }
    __syncthreads();
    if (threadIdx.x >= 1 && threadIdx.x < 7) {
        unsigned long long n = 0;
        for (int w = 0; w < waves; ++w) n += s[w * 8 + threadIdx.x];
        if (n) atomicAdd(counters + (blockIdx.x % kCounterLines) * kCounterLine + threadIdx.x, n);
    }
    if (threadIdx.x == 0 && dt_min) {
        double m = scratch[0];
        for (int w = 1; w < waves; ++w) m = fmin(m, scratch[w * 8]);
        // positive doubles order as their bit patterns; most workgroups find a
        // smaller one there already
        const unsigned long long bits = (unsigned long long)__double_as_longlong(m);
        if (m < 1e10 && bits < __hip_atomic_load(dt_min, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMin(dt_min, bits);
    }
}

}  // namespace uqk
