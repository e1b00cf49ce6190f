// closure_tile_kernel.h -- the Newton closure for systems of n = S nTotal < 64
// duals of any basis, quadrature and per-cell order, one wavefront per cell,
// FP64.  Instantiated per closure kind (closure_tile_*.hip) and per number of
// 16-row tiles that the largest order needs.
//
// Same algorithm as closure_fp64.hip (Closure::SolveClosure /
// SolveClosureSafe, closure.cpp:133-193, :297-339) with the layout of
// closure_wave_kernel.h -- Lambda, projection and Hessian as 4 x 4 x 4 FP64
// matrix products, the system in register tiles (tile_solve.h) -- at sizes
// known when it runs: loops over basis functions, points and pairs run to the
// cell's own order, and tiles past it are skipped.
//
// What bounds it: the latency of a cell's chain, as in the wave kernel.  It
// replaced a column-by-column Cholesky in LDS (closure_fp64.hip, which is
// left with the systems of 64 duals and more): Euler 2D, 65,536 cells on
// refinement levels of 12, 24 and 40 duals, 25 points, 40 time steps: 21.0 ms
// against 52.6 (26.2 with DU through the exponential and with the lane's
// numbers kept over the cell: 4 to 48 registers spilled; 22.8 with reads of 8
// bytes from LDS and tile rows skipped by branches).
#pragma once
#include <hip/hip_runtime.h>

#include "cell_queue.h"
#include "tile_solve.h"
#include "uqk_device.h"
#include "uqk_internal.h"

namespace uqk {

// LDS doubles of the workgroup's tables and of a wavefront for table width M,
// Q points and n duals at most
struct TileLds {
    int qp, ki, phiw, tables;            // row length (4 mod 8: tile_solve.h), padded basis / 4, offset of phiw, size
    int lam, lamnew, ub, du, yb, h, wave;  // offsets in a wavefront's part, and its size
    __host__ __device__ TileLds(int S, int M, int Q) {
        const int P = S * (S + 1) / 2, n = S * M;
        qp = (Q + 7) / 8 * 8 + 4;
        ki = (M + 3) / 4;
        phiw = 4 * ki * qp;
        tables = phiw + M * qp;
        lam = 0;
        lamnew = lam + n;
        ub = lamnew + n;
        du = ub + S * qp;
        yb = du + P * qp;
        h = yb + 64;
        wave = (h + (n + 1) * (n + 2) / 2 + 1) & ~1;
    }
};

template <int KIND, int NT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) newton_tile_kernel(NewtonArgs a) {
    constexpr int S = KindInfo<KIND>::S, P = S * (S + 1) / 2, PG = (P + 3) / 4;
    constexpr int DT = ((16 * NT - 1) / S + 15) / 16;  // duals per lane
    constexpr int TILES = NT * (NT + 1) / 2;
    extern __shared__ double smem[];
    const int active = a.active ? *a.active : 1;
    if (!active || (long)blockIdx.x >= a.ncell) return;
    const int M = a.M, Q = a.Q, SM = S * M;
    const TileLds at(S, M, Q);
    const int QP = at.qp;
    double* phiT = smem;             // phiT[i*QP + k]  = phi(k, i), zero past Q and M
    double* phiwT = smem + at.phiw;  // phiwT[i*QP + k] = phiw(k, i)
    for (int t = threadIdx.x; t < at.phiw; t += blockDim.x) {
        const int i = t / QP, k = t - i * QP;
        const bool in = k < Q && i < M;
        phiT[t] = in ? a.phi[k * M + i] : 0.0;
        if (i < M) phiwT[t] = in ? a.phiw[k * M + i] : 0.0;
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6;
    double* wb = smem + at.tables + wave * at.wave;
    double* Ub = wb + at.ub;
    double* DUb = wb + at.du;  // Lambda at the points (rows 0..S-1), then DU
    double* yb = wb + at.yb;
    double* H = wb + at.h;     // packed rows of the lower triangle, then the right-hand side as row n
    const ClosureParams& c = a.c;
    unsigned long long w_count[7] = {};
    double w_dt = 1e10;
    CellQueue queue((long)wave * gridDim.x + blockIdx.x, (long)gridDim.x * (blockDim.x >> 6), a.ncell, nullptr,
                    a.counter);
    for (long cell = queue.first(); cell >= 0; cell = queue.take()) {
        // (the lane's coordinates anew for each cell: what derives from them is
        // not kept in registers over the loop)
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        int p16 = lane & 15, q4 = lane >> 4;
        int s4 = (p16 & 3) < S ? (p16 & 3) : S - 1;  // this lane's state as an operand row
        queue.ask();
        // phase: inputs
        const int nt = a.nt_cell ? __builtin_amdgcn_readfirstlane(a.nt_cell[cell]) : M;
        const int n = S * nt;
        const double* ug = a.u + cell * SM;
        double* lg = a.lam + cell * SM;
        double* lam = wb + at.lam;
        double* lamnew = wb + at.lamnew;
        // dual (s, i) = (q4, p16 + 16 t) of the lane
        bool on[DT];
        double ue[DT];
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            on[t] = q4 < S && p16 + 16 * t < nt;
            ue[t] = on[t] ? ug[(p16 + 16 * t) * S + q4] : 0.0;
        }
        for (int t = lane; t < n; t += 64) lam[t] = lg[t];
        const double dx = a.uq_out && a.dt_min ? a.dx_param[cell] : 0.0;
        wave_sync();
        // phase end: inputs

        double uproj[DT];
        // ||grad L|| at the duals X (LDS): U at the points in Ub, Lambda in DUb, gradient in gout
        auto gradient = [&](const double* X, double (&gout)[DT]) -> double {
            // phase: gradient
            // W tiles of 16 points from p0 on
            auto part = [&](int p0, auto width) {
                constexpr int W = decltype(width)::value;
                double t4[4] = {0.0, 0.0, 0.0, 0.0};
                const double* ph[W];
#pragma unroll
                for (int t = 0; t < W; ++t) {
                    const int k = p0 + 16 * t + p16;
                    ph[t] = phiT + q4 * QP + (k < Q ? k : Q - 1);
                }
                in_steps<1>(
                    (nt + 3) / 4,
                    [&](int ki) {
                        Operands<W> o;
                        const int i = 4 * ki + q4;
                        o.a = i < nt ? X[i * S + s4] : 0.0;
#pragma unroll
                        for (int t = 0; t < W; ++t) o.b[t] = ph[t][4 * ki * QP];
                        return o;
                    },
                    [&](const Operands<W>& o) {
#pragma unroll
                        for (int t = 0; t < W; ++t)
                            t4[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(o.a, o.b[t], t4[t], 0, 0, 0);
                    });
#pragma unroll
                for (int t = W; t < 4; ++t) t4[t] = t4[W - 1];  // (lanes past the tiles: finite)
                group_transpose(t4);
                double U[S];
                closure_U<KIND>(c, t4, U);
                const int k = p0 + lane;
                if (k < QP) {
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        Ub[s * QP + k] = k < Q ? U[s] : 0.0;  // (an infinity times the table's zero is NaN)
                        DUb[s * QP + k] = t4[s];
                    }
                }
            };
            for (int p0 = 0; p0 < Q; p0 += 64) {
                if (Q - p0 > 32)
                    part(p0, std::integral_constant<int, 4>());
                else
                    part(p0, std::integral_constant<int, 2>());
            }
            wave_sync();
            double sq = 0.0;
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                double acc = 0.0;
                if (16 * t < (a.all_moments ? M : nt)) {
                    const int i = p16 + 16 * t < M ? p16 + 16 * t : M - 1;
                    const double *ua = Ub + s4 * QP + 2 * q4, *wa = phiwT + i * QP + 2 * q4;
                    in_steps<2>(
                        QP / 8,
                        [&](int k) {
                            Operands<1, f64x2> o;
                            o.a = two(ua + 8 * k);
                            o.b[0] = two(wa + 8 * k);
                            return o;
                        },
                        [&](const Operands<1, f64x2>& o) {
#pragma unroll
                            for (int h = 0; h < 2; ++h)
                                acc = __builtin_amdgcn_mfma_f64_4x4x4f64(o.a[h], o.b[0][h], acc, 0, 0, 0);
                        });
                }
                uproj[t] = acc;
                const double g = on[t] ? acc - ue[t] : 0.0;
                gout[t] = g;
                sq += g * g;
            }
            const double nrm = sqrt(wave_sum(sq));
            wave_sync();
            // phase end: gradient
            return nrm;
        };
        // Newton direction at the iterate of the last gradient; false if the
        // Hessian is not positive definite
        auto direction = [&](const double (&g)[DT], double (&d)[DT]) -> bool {
            // phase: hessian
            for (int k = lane; k < QP - 4; k += 64) {
                double L[S], y[P];
#pragma unroll
                for (int s = 0; s < S; ++s) L[s] = DUb[s * QP + k];
                closure_DU<KIND>(c, L, Ub[k], y);  // (the last gradient was lam's)
#pragma unroll
                for (int p = 0; p < P; ++p) DUb[p * QP + k] = y[p];
            }
            wave_sync();
            // (pairs x points)(points x state pairs), closure.cpp:255-271
            const int npair = nt * (nt + 1) / 2;
            for (int t = 0; 16 * t < npair; ++t) {
                int j, i;
                basis_pair(16 * t + p16 < npair ? 16 * t + p16 : 0, j, i);
                const double *fj = phiT + j * QP + 2 * q4, *wi = phiwT + i * QP + 2 * q4;
                const double* du[PG];
                double acc[PG];
#pragma unroll
                for (int pg = 0; pg < PG; ++pg) {
                    const int p = 4 * pg + (p16 & 3);
                    du[pg] = DUb + (p < P ? p : P - 1) * QP + 2 * q4;
                    acc[pg] = 0.0;
                }
                struct Step {
                    f64x2 f, w, d[PG];
                };
                in_steps<2>(
                    QP / 8,
                    [&](int k) {
                        Step o;
                        o.f = two(fj + 8 * k);
                        o.w = two(wi + 8 * k);
#pragma unroll
                        for (int pg = 0; pg < PG; ++pg) o.d[pg] = two(du[pg] + 8 * k);
                        return o;
                    },
                    [&](const Step& o) {
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const double av = o.f[h] * o.w[h];
#pragma unroll
                            for (int pg = 0; pg < PG; ++pg)
                                acc[pg] = __builtin_amdgcn_mfma_f64_4x4x4f64(av, o.d[pg][h], acc[pg], 0, 0, 0);
                        }
                    });
                // this lane's products: pair 16 t + 4 (p16 / 4) + q4, state pairs 4 pg + p16 % 4
                const int e = 16 * t + 4 * (p16 >> 2) + q4;
                if (e < npair) {
                    basis_pair(e, j, i);
#pragma unroll
                    for (int pg = 0; pg < PG; ++pg) {
                        const int p = 4 * pg + (p16 & 3);
                        if (p < P) {
                            const int l = p < 1 ? 0 : p < 3 ? 1 : p < 6 ? 2 : 3, m = p - l * (l + 1) / 2;
                            const int r1 = l * nt + i, r2 = l * nt + j;
                            H[r1 * (r1 + 1) / 2 + m * nt + j] = acc[pg];
                            if (m < l) H[r2 * (r2 + 1) / 2 + m * nt + i] = acc[pg];
                        }
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < DT; ++t)
                if (on[t]) H[n * (n + 1) / 2 + q4 * nt + p16 + 16 * t] = g[t];
            wave_sync();
            // phase end: hessian
            // phase: load
            f64x4 T[TILES];
#pragma unroll
            for (int tr = 0; tr < NT; ++tr)
#pragma unroll
                for (int tc = 0; tc <= tr; ++tc)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int r = 16 * tr + p16, cc = 16 * tc + 4 * e + q4;
                        const int hi = r > cc ? r : cc, lo = r > cc ? cc : r;
                        const bool in = hi <= n && lo < n;
                        const double v = H[in ? hi * (hi + 1) / 2 + lo : 0];
                        T[tile_lower(tc, tr)][e] = in ? v : 0.0;
                    }
            // phase end: load
            // phase: factor
            bool spd = false;
            static_for<NT>([&](auto last) {  // (as many tile rows as the order takes)
                constexpr int R = decltype(last)::value + 1;
                if (n >> 4 == R - 1) {
                    spd = tile_ldl<R>(T, n, p16, q4);
                    yb[lane] = tile_back<R>(T, n, p16, q4);
                }
            });
            // phase end: factor
            wave_sync();
#pragma unroll
            for (int t = 0; t < DT; ++t) d[t] = on[t] ? yb[q4 * nt + p16 + 16 * t] : 0.0;
            wave_sync();
            return spd;
        };

        double g[DT] = {}, gt[DT] = {}, d[DT] = {};
        double ng = 0.0, step = 1.0;
        int status = -1, iters = 0, halvings = 0, ngrad = 0;
        bool ub_lam = false;  // Ub and uproj belong to lam
        enum { START, TRIAL, END };
        int where = START;
        asm volatile("" : "+s"(where));  // (not cloned for its first pass)
        for (;;) {
            // (and for each pass, for the same reason)
            asm volatile("" : "+v"(lane));
            p16 = lane & 15;
            q4 = lane >> 4;
            s4 = (p16 & 3) < S ? (p16 & 3) : S - 1;
#pragma unroll
            for (int t = 0; t < DT; ++t) on[t] = q4 < S && p16 + 16 * t < nt;
            ++ngrad;
            const double nt_norm = gradient(where == TRIAL ? lamnew : lam, gt);
            if (where == END) break;
            if (where == START) {
                queue.resolve();
                ng = nt_norm;
                ub_lam = true;
                if (!c.safe && ng < c.eps) status = UQK_STATUS_CONVERGED;
            } else {
                // line search (closure.cpp:159-184): halve the step until
                // ||grad|| does not grow (SolveClosureSafe: and is finite)
                ub_lam = false;
                if (halvings > 0 && nt_norm < c.eps) {
                    status = UQK_STATUS_CONVERGED;
                } else if (halvings > 0 && halvings > c.max_halvings) {
                    status = UQK_STATUS_LINE_SEARCH;
                } else if (ng < nt_norm || (c.safe && !isfinite(nt_norm))) {
                    step *= 0.5;
                    ++halvings;
#pragma unroll
                    for (int t = 0; t < DT; ++t)
                        if (on[t]) {
                            const int f = (p16 + 16 * t) * S + q4;
                            lamnew[f] = lam[f] - step * c.alpha * d[t];
                        }
                    wave_sync();
                    continue;
                }
                if (status != UQK_STATUS_LINE_SEARCH) {
                    double* x = lam;
                    lam = lamnew;
                    lamnew = x;
                    ub_lam = true;
                    ng = nt_norm;
                    if (status < 0 && !isfinite(nt_norm)) status = UQK_STATUS_NONFINITE;
                    if (status < 0 && nt_norm < c.eps) status = UQK_STATUS_CONVERGED;
                }
            }
            if (status < 0 && iters >= c.max_iter) status = UQK_STATUS_MAX_ITERATIONS;
            if (status < 0) {
                ++iters;
#pragma unroll
                for (int t = 0; t < DT; ++t) g[t] = gt[t];
                if (!direction(g, d)) {
                    status = UQK_STATUS_NOT_SPD;
                } else if (c.max_iter == 1) {  // one-shot IPM (closure.cpp:151-154)
#pragma unroll
                    for (int t = 0; t < DT; ++t)
                        if (on[t]) lam[(p16 + 16 * t) * S + q4] -= c.alpha * d[t];
                    ub_lam = false;
                    wave_sync();
                    status = UQK_STATUS_CONVERGED;
                }
            }
            if (status < 0) {
                step = 1.0;
                halvings = 0;
#pragma unroll
                for (int t = 0; t < DT; ++t)
                    if (on[t]) {
                        const int f = (p16 + 16 * t) * S + q4;
                        lamnew[f] = lam[f] - step * c.alpha * d[t];
                    }
                wave_sync();
                where = TRIAL;
                continue;
            }
            // the outputs come from U at the returned lambda
            if (!a.uq_out || ub_lam) break;
            where = END;
        }
        // phase: outputs
        for (int t = lane; t < n; t += 64) lg[t] = lam[t];
        if (a.uq_out) {
            // uQ = U(lambda phi) (momentsolver.cpp:100) and u = <uQ phiW>
            // (:120-124); all_moments: also past the cell's order (the
            // refinement that follows cuts them at the new one)
            double* uqg = a.uq_out + cell * (long)Q * S;
            for (int t = lane; t < Q * S; t += 64) {
                const int k = t / S, s = t - k * S;
                uqg[t] = Ub[s * QP + k];
            }
#pragma unroll
            for (int t = 0; t < DT; ++t)
                if (q4 < S && p16 + 16 * t < M)
                    a.u_out[cell * SM + (p16 + 16 * t) * S + q4] = on[t] || a.all_moments ? uproj[t] : 0.0;
            if (a.dt_min) {  // momentsolver.cpp:127-133 for this cell
                double m = 1e10;
                for (int k = lane; k < Q; k += 64) {
                    double uk[S];
#pragma unroll
                    for (int s = 0; s < S; ++s) uk[s] = Ub[s * QP + k];
                    m = fmin(m, point_dt<S>(a.dtp, uk, dx));
                }
                w_dt = fmin(w_dt, wave_min(m));
            }
        }
        if (lane == 0) {
            if (a.status) a.status[cell] = status;
            if (a.iters) a.iters[cell] = iters;
        }
        w_count[1] += status != UQK_STATUS_CONVERGED ? 1ull : 0ull;
        w_count[2] += (unsigned long long)iters;
        w_count[3] += (unsigned long long)ngrad;
        wave_sync();
        // phase end: outputs
    }
    add_counts(w_count, w_dt, smem, a.counter, a.dt_min);
}

template <int KIND, int NT>
static hipError_t tile_go(const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st) {
    const TileLds at(KindInfo<KIND>::S, a.M, a.Q);
    int waves = 4;
    auto lds = [&](int w) { return sizeof(double) * ((size_t)at.tables + (size_t)w * at.wave); };
    while (waves > 1 && lds(waves) > (size_t)max_lds) waves /= 2;
    const size_t shmem = lds(waves);
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, newton_tile_kernel<KIND, NT>, 64 * waves, shmem) !=
            hipSuccess ||
        occ <= 0)
        occ = 1;
    const long want = a.ncell, cap = (long)occ * (num_cu > 0 ? num_cu : 1);
    const unsigned blocks = (unsigned)(want < cap ? (want > 0 ? want : 1) : cap);
    hipLaunchKernelGGL((newton_tile_kernel<KIND, NT>), dim3(blocks), dim3(64 * waves), shmem, st, a);
    return hipGetLastError();
}

// tiles of 16 rows that n duals and the right-hand side take
inline int tile_count(int n) { return n / 16 + 1; }

template <int KIND>
static hipError_t tile_kind(const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st) {
    switch (tile_count(KindInfo<KIND>::S * a.M)) {
        case 1: return tile_go<KIND, 1>(a, max_lds, num_cu, st);
        case 2: return tile_go<KIND, 2>(a, max_lds, num_cu, st);
        case 3: return tile_go<KIND, 3>(a, max_lds, num_cu, st);
        case 4: return tile_go<KIND, 4>(a, max_lds, num_cu, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace uqk
