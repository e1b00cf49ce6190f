// sweeps.hip -- HBM-bound sweeps of the moment solver's step body:
//   u(lambda) at the quadrature points   (momentsolver.cpp:99-101)
//   moment reconstruction u = uQ phiw    (momentsolver.cpp:120-124)
//   CFL time step, global min            (momentsolver.cpp:127-133)
//   kinetic flux + explicit Euler update (expliciteuler.cpp:8-75) with the
//     residual of the state-0 mean fused in (momentsolver.cpp:149-152)
//   mean / variance of the solution      (momentsolver.cpp:302-328)
#include <hip/hip_runtime.h>

#include "tile_solve.h"
#include "uqk_device.h"
#include "uqk_internal.h"

namespace uqk {


constexpr int kSweepThreads = 256;
constexpr int kPartialBlocks = 8192;  // grid of the grid-stride sweeps and size of the partials
// grid of the advance: its workgroups load the projection's table once each
constexpr int kAdvanceBlocks = 2048;

int sweep_partial_blocks() { return kPartialBlocks; }

// One thread per (cell, quadrature point): uq(s,k) = U_mat(sum_i lambda(s,i) phi(k,i)).
#define UQK_SKIP_IF_INACTIVE(a) \
    if ((a).active && *(a).active == 0) return;

template <int KIND>
__global__ void __launch_bounds__(kSweepThreads) eval_uq_kernel(SweepArgs a) {
    constexpr int S = KindInfo<KIND>::S;
    UQK_SKIP_IF_INACTIVE(a)
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.ncell * a.Q) return;
    long cell = t / a.Q;
    int k = (int)(t - cell * a.Q);
    int nt = a.nt_cell ? a.nt_cell[cell] : a.M;
    const double* lam = a.lam + cell * S * a.M;
    double L[S], Uv[S];
#pragma unroll
    for (int s = 0; s < S; ++s) L[s] = 0.0;
    for (int i = 0; i < nt; ++i) {
        double p = a.phi[k * a.M + i];
#pragma unroll
        for (int s = 0; s < S; ++s) L[s] += lam[i * S + s] * p;
    }
    closure_U_mat<KIND>(a.c, L, Uv);
    double* out = a.uq_out + t * S;
#pragma unroll
    for (int s = 0; s < S; ++s) out[s] = Uv[s];
}

// u(s, i) = sum_k uq(s, k) phiw(k, i) for i < nt: a wavefront's 16 / S cells
// as one FP64 matrix product (rows: cell slot x state), 16 moments at a time;
// uQ is read once, a cell's four points of a step together, and two passes'
// steps are in flight.  It is bound by that read (65,536 cells at 25 points,
// four states: 19 us; one thread per moment, every uQ read M times through
// L1, 65 us).
template <int S>
__global__ void __launch_bounds__(kSweepThreads) reconstruct_kernel(SweepArgs a) {
    constexpr int CPW = 16 / S;
    UQK_SKIP_IF_INACTIVE(a)
    const int M = a.M, Q = a.Q;
    const int lane = threadIdx.x & 63, p16 = lane & 15, q4 = lane >> 4;
    const long cell0 = ((long)blockIdx.x * (kSweepThreads / 64) + (threadIdx.x >> 6)) * CPW;
    if (cell0 >= a.ncell) return;
    const int slot = p16 / S < CPW ? p16 / S : 0;
    const long ca = cell0 + slot < a.ncell ? cell0 + slot : a.ncell - 1;
    const double* ua = a.uq + ca * S * Q + p16 % S;
    for (int ti = 0; 16 * ti < M; ++ti) {
        const int ic = 16 * ti + p16;
        const double* wb = a.phiw + (ic < M ? ic : M - 1);
        f64x4 acc = {0.0, 0.0, 0.0, 0.0};
        in_steps<4>(
            (Q + 3) / 4,
            [&](int ks) {
                Operands<1> o;
                const int k = 4 * ks + q4, kk = k < Q ? k : Q - 1;
                const double x = ua[kk * S], w = wb[kk * M];
                o.a = k < Q ? x : 0.0;
                o.b[0] = k < Q ? w : 0.0;
                return o;
            },
            [&](const Operands<1>& o) { acc = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a, o.b[0], acc, 0, 0, 0); });
        settle<18>();
#pragma unroll
        for (int e = 0; e < 4; ++e) {  // element e at (4 e + q, 16 ti + p)
            const int row = 4 * e + q4, cs = row / S;
            const long c = cell0 + cs;
            if (cs >= CPW || c >= a.ncell || ic >= M) continue;
            const int nt = a.nt_cell ? a.nt_cell[c] : M;
            a.u_out[c * S * M + ic * S + row % S] = ic < nt ? acc[e] : 0.0;
        }
    }
}

// The same with one thread per moment, for few of them over few points: a
// wavefront of reconstruct_kernel then has four cells and hardly any product
// (262,144 cells of four states: 4 moments at 5 points 38 us here, 45 there; 3
// at 3 28 and 44; 1 at 1 16 and 39; but 4 at 8 48 and 45, 3 at 12 51 and 47).
constexpr int kReconstructSmall = 32;  // moments times points below which it is taken
template <int S>
__global__ void __launch_bounds__(kSweepThreads) reconstruct_small_kernel(SweepArgs a) {
    UQK_SKIP_IF_INACTIVE(a)
    const int M = a.M, Q = a.Q;
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.ncell * S * M) return;
    const long cell = t / (S * M);
    const int e = (int)(t - cell * S * M), i = e / S, s = e - i * S;
    const int nt = a.nt_cell ? a.nt_cell[cell] : M;
    double acc = 0.0;
    if (i < nt) {
        const double* q = a.uq + cell * S * Q;
        for (int k = 0; k < Q; ++k) acc += q[k * S + s] * a.phiw[k * M + i];
    }
    a.u_out[t] = acc;
}

// MomentSolver refinement (momentsolver.cpp:104-117) with ComputeRefIndicator
// (:271-289), one thread per cell.  The indicator of a cell at level l is
// |u(0, nt-1)| + |u(0, nt-2)| for one uncertain dimension, else the sum of
// |u(0, i)| over the moments the level adds (i from nTotal(l-1), or from 1 at
// level 0).  Above refine_above the cell moves up a level, below
// coarsen_below down, and never above max_level (the cap of refinement
// retardation).  A cell whose nt_cell is no level's nTotal is left alone.
__global__ void __launch_bounds__(kSweepThreads) refine_kernel(RefineArgs a) {
    UQK_SKIP_IF_INACTIVE(a)
    const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= a.ncell) return;
    const int nt = a.nt_cell[j];
    int lev = -1;
    for (int l = 0; l < a.nlev; ++l)
        if (a.nt_level[l] == nt) lev = l;
    if (lev < 0) return;
    const double* u = a.u + j * a.S * a.M;
    double ind = 0.0;
    if (a.dim_xi == 1) {
        ind = fabs(u[(nt - 1) * a.S]);
        if (nt >= 2) ind += fabs(u[(nt - 2) * a.S]);
    } else {
        for (int i = lev == 0 ? 1 : a.nt_level[lev - 1]; i < nt; ++i) ind += fabs(u[i * a.S]);
    }
    if (ind > a.refine_above && lev < a.nlev - 1)
        ++lev;
    else if (ind < a.coarsen_below && lev > 0)
        --lev;
    if (lev > a.max_level) lev = a.max_level;
    a.nt_cell[j] = a.nt_level[lev];
}

__device__ __forceinline__ double block_min(double v) {
    __shared__ double red[kSweepThreads / 64];
    v = wave_min(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = fmin(r, red[w]);
    __syncthreads();
    return r;
}

__device__ __forceinline__ double block_sum(double v) {
    __shared__ double red[kSweepThreads / 64];
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r += red[w];
    __syncthreads();
    return r;
}

// Per-block minimum of ComputeDt over cells (grid-stride), then a one-block finish.
template <int KIND>
__global__ void __launch_bounds__(kSweepThreads) dt_partial_kernel(SweepArgs a) {
    constexpr int S = KindInfo<KIND>::S;
    UQK_SKIP_IF_INACTIVE(a)
    double m = 1e10;
    for (long cell = (long)blockIdx.x * blockDim.x + threadIdx.x; cell < a.ncell; cell += (long)gridDim.x * blockDim.x) {
        const double* q = a.uq + cell * S * a.Q;
        double dx = a.dx_param[cell];
        for (int k = 0; k < a.Q; ++k) m = fmin(m, point_dt<S>(a.p, q + k * S, dx));
    }
    m = block_min(m);
    if (threadIdx.x == 0) a.partial[blockIdx.x] = m;
}

__global__ void __launch_bounds__(kSweepThreads) min_finish_kernel(SweepArgs a) {
    UQK_SKIP_IF_INACTIVE(a)
    double m = 1e10;
    for (int t = threadIdx.x; t < a.npartial; t += blockDim.x) m = fmin(m, a.partial[t]);
    m = block_min(m);
    if (threadIdx.x == 0) *a.scalar_out = m;
}

__global__ void __launch_bounds__(kSweepThreads) sum_finish_kernel(SweepArgs a) {
    UQK_SKIP_IF_INACTIVE(a)
    double m = 0.0;
    for (int t = threadIdx.x; t < a.npartial; t += blockDim.x) m += a.partial[t];
    m = block_sum(m);
    if (threadIdx.x == 0) *a.scalar_out = m;
}

// Cells per wavefront of the advance: lanes take (cell slot, quadrature
// point) for Q <= 32, as many cells as 64 lanes and the 16 rows of one MFMA
// tile (cells x states) allow; one cell with ceil(Q/64) points per lane else.
__host__ __device__ inline int advance_cells_per_wave(int S, int Q) {
    if (Q > 32) return 1;
    const int by_lanes = 64 / Q, by_rows = 16 / S;
    return by_lanes < by_rows ? by_lanes : by_rows;
}

// LDS doubles per wavefront of the advance: the edge-summed point fluxes of
// its cells, (cell slot, point, state).
__host__ __device__ inline int advance_wave_doubles(int S, int Q) {
    return advance_cells_per_wave(S, Q) * Q * S;
}

// a read-only value at a uniform address, through the scalar cache
template <class T> __device__ __forceinline__ T uniform_load(const T* p) {
    return *(const __attribute__((address_space(4))) T*)p;
}

// ExplicitEuler::Advance (expliciteuler.cpp:8-75) with numFlux
// (momentsolver.cpp:413-416) for a wavefront's cells: each lane owns a
// quadrature point of one cell and sums the point fluxes of all the cell's
// edges in registers, in edge order (the projection onto phiw is linear, so
// the edges share one projection); the shallow-water bed friction enters as
// -area * S(u) at the point before the projection; the projection
// rhs(s, i) = sum_k G(s, k) phiW(k, i) of all the wave's cells is one FP64
// matrix product (rows: cell slot x state), and the lanes holding its elements
// update the moments.  The residual |u_new(0,0) - u_old(0,0)| * area is
// accumulated per block.
// What bounds it: the wait for memory at four wavefronts per SIMD (60% of
// their time), and the fluxes' instructions (half of the SIMDs' time).  uQ is
// read from HBM once (62 MB of 65,536 cells at 25 points and four states).
// Reciprocals and roots as refined estimates and the cell's own state formed
// once for its edges, edge data in one load per vector or (ONE) in scalar
// registers, 2,048 workgroups instead of 8,192 that each load the projection's
// table: 94 -> 79 us there, 777 -> 466 us for 65,536 cells at 125 points and
// three states, whose projection took 16-row products for 3 rows.
// ONE: a wavefront has one cell (Q > 32).  The cell, its edges and their
// normals are then uniform, in scalar registers.
// (four waves per SIMD: the kernel waits on memory, and the register budget
// of four waves holds it)
template <int KIND, bool ONE>
__global__ void __launch_bounds__(kSweepThreads) __attribute__((amdgpu_waves_per_eu(4))) advance_kernel(SweepArgs a) {
    constexpr int S = KindInfo<KIND>::S;
    UQK_SKIP_IF_INACTIVE(a)
    extern __shared__ double smem[];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int M = a.M, Q = a.Q, SM = S * M, E = a.nedge, D = a.dim;
    const int CPW = ONE ? 1 : advance_cells_per_wave(S, Q);
    double* Gs = smem + wave * advance_wave_doubles(S, Q);
    const bool wlds = a.table_lds != 0;
    double* wt = smem + (blockDim.x >> 6) * advance_wave_doubles(S, Q);
    if (wlds) {
        for (int t = threadIdx.x; t < Q * M; t += blockDim.x) wt[t] = a.phiw[t];
        __syncthreads();
    }
    const double* phiw = wlds ? wt : a.phiw;
    const double dt = a.dt_dev ? *a.dt_dev : a.dt;
    const bool fric = (S == 3 && a.p.problem == UQK_SHALLOW_WATER2D_PROBLEM && a.p.friction > 0.0);
    // this lane's cell slot and first point
    const int slot = ONE ? 0 : lane / Q;
    const int k0 = ONE ? lane : lane - slot * Q;
    const bool lane_on = slot < CPW && k0 < Q;
    double res = 0.0;
    const long nwaves = (long)gridDim.x * (blockDim.x >> 6);
    for (long cell0 = ((long)blockIdx.x * (blockDim.x >> 6) + wave) * CPW; cell0 < a.ncell; cell0 += nwaves * CPW) {
        const long cell = ONE ? (long)__builtin_amdgcn_readfirstlane((int)cell0) : cell0 + slot;
        const bool on = lane_on && cell < a.ncell;
        int bc = UQK_BC_DIRICHLET;
        if constexpr (ONE)
            bc = uniform_load(a.bc + cell);
        else if (on)
            bc = a.bc[cell];
        if (on && bc != UQK_BC_DIRICHLET) {
            const double* uqj = a.uq + cell * S * Q;
            const bool wall = (bc == UQK_BC_NOSLIP || bc == UQK_BC_SWWALL);
            const double area = ONE ? uniform_load(a.area + cell) : a.area[cell];
            int nb[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                nb[e] = 0;
                if (e < E) nb[e] = ONE ? uniform_load(a.nbr + cell * E + e) : a.nbr[cell * E + e];
            }
            for (int k = k0; k < Q; k += 64) {
                double uj[S], Gsum[S], v[S], vn[S];
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    uj[s] = uqj[k * S + s];
                    Gsum[s] = 0.0;
                }
                // an edge's other state, with ONE sent for before the edge before
                // it is used (without, the registers are worth more: 98 us
                // against 109 with it, 65,536 cells of four states at 25 points;
                // the reference reads the never-written uQ[nCells], zero)
                auto other = [&](int j, double (&x)[S]) {
                    const double* src = j != a.ncell ? a.uq + (long)j * Q * S : uqj;
#pragma unroll
                    for (int s = 0; s < S; ++s) x[s] = src[k * S + s];
                };
                if constexpr (ONE) other(nb[0], v);
                const PointState pj = point_state<S>(a.p, uj);
#pragma unroll 1
                for (int e = 0; e < E; ++e) {
                    const int nbe = e < 2 ? (e == 0 ? nb[0] : nb[1]) : (e == 2 ? nb[2] : nb[3]);
                    if constexpr (!ONE) other(nbe, vn);
                    if (ONE && e + 1 < E) other(e == 0 ? nb[1] : e == 1 ? nb[2] : nb[3], vn);
                    const double* nu = a.unit_normal + (cell * E + e) * D;
                    const double* nv = a.normal + (cell * E + e) * D;
                    double nux, nuy = 0.0, nx, ny = 0.0;
                    if constexpr (ONE) {
                        nux = uniform_load(nu);
                        nx = uniform_load(nv);
                        if (D > 1) {
                            nuy = uniform_load(nu + 1);
                            ny = uniform_load(nv + 1);
                        }
                    } else if (D > 1) {
                        const f64x2 u2 = two(nu), v2 = two(nv);
                        nux = u2[0];
                        nuy = u2[1];
                        nx = v2[0];
                        ny = v2[1];
                    } else {
                        nux = nu[0];
                        nx = nv[0];
                    }
                    const bool edge = nbe == a.ncell;
                    double l[S], r[S], G[S];
                    PointState pl = pj;
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        l[s] = uj[s];
                        r[s] = edge ? 0.0 : ONE ? v[s] : vn[s];
                    }
                    if (edge && wall) {
                        // ghost state: velocity reflected to the tangential
                        // part (expliciteuler.cpp:25-58); the flux is G(ghost, ghost)
                        if constexpr (S >= 3) {
                            const double bx = a.bnormal[cell * D + 0], by = a.bnormal[cell * D + 1];
                            const double rho = uj[0], vx = uj[1] / rho, vy = uj[2] / rho;
                            const double vn = bx * vx + by * vy;
                            const double tx = vx - vn * bx, ty = vy - vn * by;
                            if constexpr (S == 4) {
                                if (bc == UQK_BC_NOSLIP) l[3] += rho * 0.5 * ((tx * tx + ty * ty) - (vx * vx + vy * vy));
                            }
                            l[1] = rho * tx;
                            l[2] = rho * ty;
                        }
#pragma unroll
                        for (int s = 0; s < S; ++s) r[s] = l[s];
                        pl = point_state<S>(a.p, l);
                    }
                    point_flux<S>(a.p, l, pl, r, point_state<S>(a.p, r), nux, nuy, nx, ny, G);
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        Gsum[s] += G[s];
                        v[s] = vn[s];
                    }
                }
                if (fric) {
                    // bed friction S_s = -cf |v| q_s / h (s = 1, 2) at this point
                    const double cf =
                        a.p.friction * (1.0 + (a.p.friction_dim >= 0 ? a.xi[k * a.d + a.p.friction_dim] : 0.0));
                    const double hi = recip_any(uj[0]);
                    const double sp = sqrt_f64(uj[1] * uj[1] + uj[2] * uj[2]) * hi;
#pragma unroll
                    for (int s = 1; s < S; ++s) Gsum[s] += area * (cf * sp * uj[s] * hi);
                }
#pragma unroll
                for (int s = 0; s < S; ++s) Gs[(slot * Q + k) * S + s] = Gsum[s];
            }
        }
        wave_sync();
        // projection and update: D = A B with A(r, k) = G(cell slot r / S,
        // state r % S, point k) and B(k, i) = phiW(k, i); the lanes that hold
        // D(r, i) update the moment
        const int p16 = lane & 15, q4 = lane >> 4;
        const int ar = ONE ? p16 & 3 : p16, ar_slot = ar / S < CPW ? ar / S : 0;
        const double* ga = Gs + ar_slot * Q * S + ar % S;
        const bool ar_on = ONE ? ar < S && bc != UQK_BC_DIRICHLET
                               : ar / S < CPW && cell0 + ar_slot < a.ncell &&
                                     a.bc[cell0 + ar_slot] != UQK_BC_DIRICHLET;
        // row r, column ic of D, with the moment's value us and its old one
        auto update = [&](int row, int ic, double acc, double us, double old) {
            const int cs = row / S, st = row - cs * S, f = ic * S + st;
            const long c = cell0 + cs;
            if (cs >= CPW || c >= a.ncell || ic >= M) return;
            const int nt = !a.nt_cell ? M : ONE ? uniform_load(a.nt_cell + cell) : a.nt_cell[c];
            const int bcc = ONE ? bc : a.bc[c];
            const double ac = ONE ? uniform_load(a.area + cell) : a.area[c];
            double v = us;
            if (a.cut && ic >= nt) {  // past the order that the refinement chose
                v = 0.0;
                a.cut[c * SM + f] = 0.0;
            }
            if (bcc != UQK_BC_DIRICHLET && ic < nt) v -= (dt / ac) * acc;
            a.u_out[c * SM + f] = v;
            if (f == 0) res += fabs(v - old) * ac;
        };
        for (int ti = 0; 16 * ti < M; ++ti) {
            const int ic = 16 * ti + p16;
            const double* wb = phiw + (ic < M ? ic : M - 1);
            auto load = [&](int ks) {
                Operands<1> o;
                const int k = 4 * ks + q4, kk = k < Q ? k : Q - 1;
                const double x = ga[kk * S];
                o.a = ar_on && k < Q ? x : 0.0;
                o.b[0] = wb[kk * M];
                return o;
            };
            // u: reconstructed moments; u_out: in the previous moments, out the new
            if constexpr (ONE) {
                // S <= 4 rows: 4 x 4 x 4 products (16 x 16 x 4 ones take four
                // times as long); lane 16 q + p gets D(q, 16 ti + p)
                const long f = cell0 * SM + ic * S + q4;
                const bool has = q4 < S && ic < M && cell0 < a.ncell;
                const double us = has ? a.u[f] : 0.0, old = has ? a.u_out[f] : 0.0;
                double acc = 0.0;
                in_steps<4>((Q + 3) / 4, load, [&](const Operands<1>& o) {
                    acc = __builtin_amdgcn_mfma_f64_4x4x4f64(o.a, o.b[0], acc, 0, 0, 0);
                });
                update(q4, ic, acc, us, old);
            } else {
                f64x4 acc = {0.0, 0.0, 0.0, 0.0};
                for (int ks = 0; ks < (Q + 3) / 4; ++ks) {
                    const Operands<1> o = load(ks);
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a, o.b[0], acc, 0, 0, 0);
                }
                settle<18>();
#pragma unroll
                for (int e = 0; e < 4; ++e) {  // element e at (4 e + q, 16 ti + p)
                    const int row = 4 * e + q4, cs = row / S;
                    const long f = (cell0 + cs) * SM + ic * S + row - cs * S;
                    const bool has = cs < CPW && cell0 + cs < a.ncell && ic < M;
                    update(row, ic, acc[e], has ? a.u[f] : 0.0, has ? a.u_out[f] : 0.0);
                }
            }
        }
        wave_sync();
    }
    __syncthreads();
    res = block_sum(res);
    if (threadIdx.x == 0) a.partial[blockIdx.x] = res;
}

// sum over the SUB lanes (32 or 64) that share a cell, in every lane
template <int SUB> __device__ __forceinline__ double sub_sum(double v) {
    v = row_sum(v);
    if constexpr (SUB == 64) return group_sum(v);
    const long long x = __double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)x, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(x >> 32), false, false);
    return __longlong_as_double(((long long)hi[0] << 32) | (unsigned)lo[0]) +
           __longlong_as_double(((long long)hi[1] << 32) | (unsigned)lo[1]);
}

// E and Var of each state from the closure at lambda (WriteMeanAndVar,
// momentsolver.cpp:302-328): lanes over quadrature points (up to 128 per
// cell), the two weighted sums over them by DPP and row swaps.  A wavefront
// has two cells where they have 32 points or fewer, else one.  Bound by the
// loads of the duals and the closure's exponentials: 65,536 cells at 25
// points, four states: 42 us (108 with one cell per wavefront, U formed
// for a second point that no lane had, and sums through LDS).
template <int KIND, int SUB>
__global__ void __launch_bounds__(kSweepThreads) mean_var_kernel(SweepArgs a) {
    constexpr int S = KindInfo<KIND>::S;
    constexpr int KP = SUB == 64 ? 2 : 1;  // quadrature points per lane
    constexpr int CPW = 64 / SUB;
    const int lane = threadIdx.x & (SUB - 1), half = (threadIdx.x & 63) / SUB;
    const long step = (long)gridDim.x * (blockDim.x >> 6) * CPW;
    for (long cell0 = ((long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * CPW; cell0 < a.ncell;
         cell0 += step) {
        const bool has = cell0 + half < a.ncell;
        const long cell = has ? cell0 + half : cell0;
        const int nt = a.nt_cell ? a.nt_cell[cell] : a.M;
        const double* lam = a.lam + cell * S * a.M;
        double Uv[KP][S], w0[KP];
#pragma unroll
        for (int h = 0; h < KP; ++h) {
            const int k = lane + SUB * h;
#pragma unroll
            for (int s = 0; s < S; ++s) Uv[h][s] = 0.0;  // (U of Lambda = 0 may be NaN)
            w0[h] = 0.0;
            if (k < a.Q) {
                double L[S];
#pragma unroll
                for (int s = 0; s < S; ++s) L[s] = 0.0;
                const double* ph = a.phi + k * a.M;
#pragma unroll 4
                for (int i = 0; i < nt; ++i) {
                    const double p = ph[i];
#pragma unroll
                    for (int s = 0; s < S; ++s) L[s] += lam[i * S + s] * p;
                }
                w0[h] = a.phiw[k * a.M + 0];
                closure_U<KIND>(a.c, L, Uv[h]);
            }
        }
        double E[S], V[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            double e = 0.0;
#pragma unroll
            for (int h = 0; h < KP; ++h) e += Uv[h][s] * w0[h];
            E[s] = sub_sum<SUB>(e);
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
            double v = 0.0;
#pragma unroll
            for (int h = 0; h < KP; ++h) v += (Uv[h][s] - E[s]) * (Uv[h][s] - E[s]) * w0[h];
            V[s] = sub_sum<SUB>(v);
        }
        if (lane == 0 && has) {
            double* out = a.mv_out + cell * 2 * S;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                out[s] = E[s];
                out[S + s] = V[s];
            }
        }
    }
}

// The end of a replayed step: residual and t (momentsolver.cpp:134-152), run
// totals, and what the next step's launches need (zero closure counters, the
// start value 1e10 of ComputeDt's MIN, the active flag: t < t_end and steps <
// max_steps and no failed cell; set_recon: the step's closure left its outputs
// at the current lambda for every cell).  One workgroup: what it costs is
// latency, so all loads are sent at once (10.8 us per step with 256 threads
// over 8,192 partials).
constexpr int kEndThreads = 1024;
__global__ void __launch_bounds__(kEndThreads) step_end_kernel(RunState* rs, double* scalars,
                                                               unsigned long long* counters,
                                                               const double* partial, int npartial, int set_recon) {
    __shared__ unsigned long long total[kCounterLine];
    __shared__ double red[kEndThreads / 64];
    const int t = threadIdx.x;
    const int active = rs->active;
    const unsigned long long mine = t < kClosureCounters ? counters[t] : 0ull;
    double v[kPartialBlocks / kEndThreads];
#pragma unroll
    for (int i = 0; i < kPartialBlocks / kEndThreads; ++i) {
        const int at = t + i * kEndThreads;
        v[i] = at < npartial ? partial[at] : 0.0;
    }
    if (!active) return;
    if (t < kCounterLine) total[t] = 0ull;
    __syncthreads();
    if (mine) atomicAdd(&total[t % kCounterLine], mine);
    double m = 0.0;
#pragma unroll
    for (int i = 0; i < kPartialBlocks / kEndThreads; ++i) m += v[i];
    m = wave_sum(m);
    if ((t & 63) == 0) red[t >> 6] = m;
    if (t < kClosureCounters) counters[t] = 0ull;
    __syncthreads();
    if (t == 0) {
        m = red[0];
        for (int w = 1; w < kEndThreads / 64; ++w) m += red[w];
        const double time = rs->t + scalars[0];
        const long long steps = rs->steps + 1;
        const long long nfail = rs->nfail + (long long)total[1];
        rs->t = time;
        rs->residual = m;
        rs->steps = steps;
        rs->nfail = nfail;
        rs->newton += (long long)total[2];
        rs->gradients += (long long)total[3];
        rs->factorizations += (long long)total[5];
        rs->reuse_steps += (long long)total[6];
        scalars[0] = 1e10;
        rs->active = (time < rs->t_end && (rs->max_steps < 0 || steps < rs->max_steps) && nfail == 0) ? 1 : 0;
        if (set_recon) rs->recon = 1;
    }
}

hipError_t launch_step_end(RunState* rs, double* scalars, unsigned long long* counters, const double* partial,
                           int set_recon, int npartial, hipStream_t st) {
    hipLaunchKernelGGL(step_end_kernel, dim3(1), dim3(kEndThreads), 0, st, rs, scalars, counters, partial, npartial,
                       set_recon);
    return hipGetLastError();
}

__global__ void fill_u64_kernel(unsigned long long* p, int n) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = 0ull;
}

__global__ void fill_f64_kernel(double* p, int n, double v) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
#define UQK_DISPATCH(kind, FN, ...)                                                                     \
    switch (kind) {                                                                                     \
        case UQK_BOUNDED_BARRIER: FN<UQK_BOUNDED_BARRIER>(__VA_ARGS__); break;                         \
        case UQK_EULER1D: FN<UQK_EULER1D>(__VA_ARGS__); break;                                         \
        case UQK_EULER2D: FN<UQK_EULER2D>(__VA_ARGS__); break;                                         \
        case UQK_SHALLOW_WATER2D: FN<UQK_SHALLOW_WATER2D>(__VA_ARGS__); break;                         \
        case UQK_SHALLOW_WATER2D_BARRIER: FN<UQK_SHALLOW_WATER2D_BARRIER>(__VA_ARGS__); break;         \
        default: return hipErrorInvalidValue;                                                           \
    }

template <int KIND> static void go_eval_uq(const SweepArgs& a, hipStream_t st) {
    long total = a.ncell * a.Q;
    int blocks = (int)((total + kSweepThreads - 1) / kSweepThreads);
    hipLaunchKernelGGL(eval_uq_kernel<KIND>, dim3(blocks), dim3(kSweepThreads), 0, st, a);
}
hipError_t launch_eval_uq(int kind, const SweepArgs& a, hipStream_t st) {
    if (a.ncell <= 0) return hipSuccess;
    UQK_DISPATCH(kind, go_eval_uq, a, st);
    return hipGetLastError();
}

hipError_t launch_refine(const RefineArgs& a, hipStream_t st) {
    if (a.ncell <= 0) return hipSuccess;
    const int blocks = (int)((a.ncell + kSweepThreads - 1) / kSweepThreads);
    hipLaunchKernelGGL(refine_kernel, dim3(blocks), dim3(kSweepThreads), 0, st, a);
    return hipGetLastError();
}

template <int S> static void go_reconstruct(const SweepArgs& a, hipStream_t st) {
    const bool few = a.M * a.Q < kReconstructSmall;
    // work items (moments or cells) per workgroup
    const long items = few ? a.ncell * S * a.M : a.ncell, per = few ? kSweepThreads : (kSweepThreads / 64) * (16 / S);
    const dim3 blocks((unsigned)((items + per - 1) / per));
    if (few)
        hipLaunchKernelGGL(reconstruct_small_kernel<S>, blocks, dim3(kSweepThreads), 0, st, a);
    else
        hipLaunchKernelGGL(reconstruct_kernel<S>, blocks, dim3(kSweepThreads), 0, st, a);
}
hipError_t launch_reconstruct(const SweepArgs& a, hipStream_t st) {
    if (a.ncell <= 0) return hipSuccess;
    switch (a.S) {
        case 1: go_reconstruct<1>(a, st); break;
        case 3: go_reconstruct<3>(a, st); break;
        case 4: go_reconstruct<4>(a, st); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

static int dt_blocks(long ncell) {
    const long want = (ncell + kSweepThreads - 1) / kSweepThreads;
    return (int)(want < 1 ? 1 : (want < kPartialBlocks ? want : kPartialBlocks));
}
template <int KIND> static void go_dt(const SweepArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(dt_partial_kernel<KIND>, dim3(dt_blocks(a.ncell)), dim3(kSweepThreads), 0, st, a);
}
hipError_t launch_dt(int kind, const SweepArgs& a, hipStream_t st) {
    UQK_DISPATCH(kind, go_dt, a, st);
    SweepArgs b = a;
    b.npartial = dt_blocks(a.ncell);
    hipLaunchKernelGGL(min_finish_kernel, dim3(1), dim3(kSweepThreads), 0, st, b);
    return hipGetLastError();
}

// Workgroups of the advance, each of which leaves one partial residual: as
// many as the cells fill, up to kPartialBlocks (a small mesh that launches and
// sums all of them spends 20 us of its step on that).
int advance_partials(int S, int Q, long ncell) {
    const long per = (long)advance_cells_per_wave(S, Q) * (kSweepThreads / 64);
    const long want = (ncell + per - 1) / per;
    return (int)(want < 1 ? 1 : (want < kAdvanceBlocks ? want : kAdvanceBlocks));
}

template <int KIND> static void go_advance(const SweepArgs& a, hipStream_t st) {
    constexpr int S = KindInfo<KIND>::S;
    size_t shmem = sizeof(double) * (kSweepThreads / 64) * advance_wave_doubles(S, a.Q);
    SweepArgs b = a;
    // PhiW goes to LDS while a workgroup stays within 64 KB
    b.table_lds = shmem + sizeof(double) * a.Q * a.M <= 65536;
    if (b.table_lds) shmem += sizeof(double) * a.Q * a.M;
    const dim3 blocks(advance_partials(S, a.Q, a.ncell));
    if (advance_cells_per_wave(S, a.Q) == 1)
        hipLaunchKernelGGL((advance_kernel<KIND, true>), blocks, dim3(kSweepThreads), shmem, st, b);
    else
        hipLaunchKernelGGL((advance_kernel<KIND, false>), blocks, dim3(kSweepThreads), shmem, st, b);
}
hipError_t launch_advance(int kind, const SweepArgs& a, hipStream_t st) {
    UQK_DISPATCH(kind, go_advance, a, st);
    return hipGetLastError();
}

hipError_t launch_residual(const SweepArgs& a, hipStream_t st) {
    SweepArgs b = a;
    b.npartial = advance_partials(a.S, a.Q, a.ncell);
    hipLaunchKernelGGL(sum_finish_kernel, dim3(1), dim3(kSweepThreads), 0, st, b);
    return hipGetLastError();
}

template <int KIND> static void go_mean_var(const SweepArgs& a, hipStream_t st) {
    const long per = (kSweepThreads / 64) * (a.Q <= 32 ? 2 : 1);
    const long want = (a.ncell + per - 1) / per;
    const dim3 blocks((unsigned)(want < kPartialBlocks ? want : kPartialBlocks));
    if (a.Q <= 32)
        hipLaunchKernelGGL((mean_var_kernel<KIND, 32>), blocks, dim3(kSweepThreads), 0, st, a);
    else
        hipLaunchKernelGGL((mean_var_kernel<KIND, 64>), blocks, dim3(kSweepThreads), 0, st, a);
}
hipError_t launch_mean_var(int kind, const SweepArgs& a, hipStream_t st) {
    if (a.ncell <= 0) return hipSuccess;
    if (a.Q > 128) return hipErrorInvalidValue;  // two quadrature points per lane
    UQK_DISPATCH(kind, go_mean_var, a, st);
    return hipGetLastError();
}

hipError_t launch_fill_f64(double* p, int n, double v, hipStream_t st) {
    hipLaunchKernelGGL(fill_f64_kernel, dim3((n + 63) / 64), dim3(64), 0, st, p, n, v);
    return hipGetLastError();
}

hipError_t launch_fill_u64(unsigned long long* p, int n, hipStream_t st) {
    hipLaunchKernelGGL(fill_u64_kernel, dim3((n + 63) / 64), dim3(64), 0, st, p, n);
    return hipGetLastError();
}

}  // namespace uqk
