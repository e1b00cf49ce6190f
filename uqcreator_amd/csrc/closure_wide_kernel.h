// closure_wide_kernel.h -- the Newton closure for systems of n = S nTotal >= 64
// duals, up to 127 with four states and 111 with fewer (wide_limit), of any
// basis, quadrature and per-cell order, one wavefront per cell and one
// wavefront per SIMD: the whole system, up to 36 tiles of 16 x 16 doubles,
// lies in that wavefront's 512 registers.
// Instantiated per closure kind (closure_wide_*.hip) and per number of
// 16-row tiles that the largest order needs.
//
// Same algorithm as closure_block.hip (Closure::SolveClosure /
// SolveClosureSafe, closure.cpp:133-193, :297-339) with the layout of
// closure_tile_kernel.h.  Unknowns in the order of the duals, r = i S + s.
//   * Hessian (closure.cpp:255-271): (pairs x points)(points x state pairs) as
//     4 x 4 x 4 FP64 matrix products, 32 basis pairs at a time in the order of
//     their rows; the rows go through a ring of some rows in LDS into the
//     tiles, four at a time, so that LDS holds a window of the matrix only;
//   * factorisation and solve, or the explicit inverse where the time loop
//     keeps it: tile_solve.h;
//   * the time loop's mixed closure keeps the inverse P of each cell's last
//     Hessian, rounded to FP32, in a per-cell slot (lower tiles, each lane's
//     four entries in a run): while it stays good, the next steps' Newton
//     steps take d = P g + P (g - H P g) against the FP64 Hessian-vector
//     product, with no Hessian and no factorisation.
//
// What bounds it: instruction and matrix issue of the one wavefront.  Cycles
// at n = 105, 125 points (shallow water, barrier): Hessian 120 K (43 K of it
// the 2,560 4 x 4 x 4 products), sweep 115 K (48 K the 756 16 x 16 x 4
// products), gradient 7.6 K, product with the kept inverse 7.1 K (1.5 of every
// 4 instructions convert it from FP32), Hessian-vector product 7.8 K.  A
// workgroup of four wavefronts per cell (closure_block.hip), two resident per
// CU, takes 75 K, 149 K and 18 K for the first three, which is four to nine
// times as much per wavefront and cell: 65,536 cells of the dam break, 12 time
// steps: 31 ms against 89.  Orders of 12 to 112 duals, 49 points, 16,384 cells,
// 12 steps: 9.2 ms against 28.  The workgroup kernel is left with more duals,
// and with the sizes at which newton_wide_takes finds it faster.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "cell_queue.h"
#include "tile_solve.h"
#include "uqk_device.h"
#include "uqk_internal.h"

namespace uqk {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// tiles of 16 rows that n duals and the right-hand side take
__host__ __device__ constexpr int wide_tiles(int n) { return n / 16 + 1; }

// floats of a cell's kept inverse: the lower tiles of the rows that n duals
// take (without the right-hand side's)
__host__ __device__ constexpr long wide_kept(int n) {
    const long r = (n + 15) / 16;
    return 256 * (r * (r + 1) / 2);
}

// Largest system: 127 duals and the right-hand side are eight tile rows; with
// fewer than four states a lane holds more duals of every vector, for which
// the registers beside that many tiles do not last.
__host__ __device__ constexpr int wide_limit(int states) { return states < 4 ? 111 : 127; }

// LDS doubles of the workgroup's tables and of a wavefront for table width M,
// Q points and S M duals at most
struct WideLds {
    int qp, ki, phiw, tables;                  // row length, padded basis / 4, offset of phiw, size
    int lam, lamnew, ub, du, yb, ring, wave;   // offsets in a wavefront's part, and its size
    __host__ __device__ WideLds(int S, int M, int Q, int ring_size) {
        const int P = S * (S + 1) / 2, n = S * M;
        // (4 mod 8: f64x2 reads of sixteen rows fall on all banks once)
        qp = (Q + 7) / 8 * 8 + 4;
        ki = (M + 3) / 4;
        phiw = 4 * ki * qp;
        tables = phiw + M * qp;
        lam = 0;
        lamnew = lam + n;
        ub = lamnew + n;
        du = ub + S * qp;
        yb = du + P * qp;
        ring = yb + 128;
        const int r = ring_size + n;  // a row that starts in the ring may run past its end
        wave = (ring + (r > 512 ? r : 512) + 1) & ~1;
    }
};

// Length of the ring: the packed rows from a group of four on that the basis
// pairs up to the last one the group needs, and 31 more, fill
inline int wide_ring(int S, int M) {
    const int n = S * M, npair = M * (M + 1) / 2;
    int most = 0, done = 0;
    for (int r0 = 0; r0 < n; r0 += 4) {
        const int i = (r0 + 3) / S < M ? (r0 + 3) / S : M - 1;
        while (done < (i + 1) * (i + 2) / 2) done += 32;
        const int last = (done < npair ? done : npair) - 1;
        int il = 0;
        while ((il + 1) * (il + 2) / 2 <= last) ++il;
        const int end = S * (il + 1);
        const int span = end * (end + 1) / 2 - r0 * (r0 + 1) / 2;
        most = span > most ? span : most;
    }
    return most;
}

template <int KIND, int NT, bool KEEP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) newton_wide_kernel(NewtonArgs a) {
    constexpr int S = KindInfo<KIND>::S, P = S * (S + 1) / 2, PG = (P + 3) / 4;
    constexpr int DT = ((16 * NT - 1) / S + 15) / 16;  // duals per lane
    constexpr int TILES = NT * (NT + 1) / 2;
    extern __shared__ double smem[];
    const int active = a.active ? *a.active : 1;
    if (!active) return;
    const long ncells = a.cell_list ? (long)*a.cell_count : a.ncell;
    if ((long)blockIdx.x >= ncells) return;
    const int M = a.M, Q = a.Q, SM = S * M, RS = a.wave_doubles;
    const WideLds at(S, M, Q, RS);
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
    double* yb = wb + at.yb;   // a vector over the unknowns, zero past n
    double* ring = wb + at.ring;
    const ClosureParams& c = a.c;
    int lane, p16, q4, s4;  // s4: this lane's state as an operand row
    // (the lane's coordinates anew for each cell and pass: what derives from
    // them is not kept in registers over the loop)
    auto renew = [&]() {
        lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        p16 = lane & 15;
        q4 = lane >> 4;
        s4 = (p16 & 3) < S ? (p16 & 3) : S - 1;
    };
    renew();
    unsigned long long w_count[7] = {};
    double w_dt = 1e10;
    CellQueue queue((long)wave * gridDim.x + blockIdx.x, (long)gridDim.x * (blockDim.x >> 6), ncells, a.cell_list,
                    a.counter);
    // a cell's inputs, sent for while the cell before it computes and waited
    // for before that one's results are stored; the kept inverse follows them,
    // still before the stores
    double u_n[DT] = {}, l_n[DT] = {}, g_n[DT] = {}, dx_n = 0.0;
    int nt_n = M, tag_n = 0;
    auto prefetch = [&](long cl) {
        if (cl < 0) return;
        nt_n = a.nt_cell ? a.nt_cell[cl] : M;
        tag_n = a.pinv_mode == 1 && cl < a.pinv_slots ? a.pinv_ok[cl] : 0;
        if (a.uq_out && a.dt_min) dx_n = a.dx_param[cl];
#pragma unroll
        for (int t = 0; t < DT; ++t)
            if (q4 < S && p16 + 16 * t < M) {
                const long f = cl * SM + (p16 + 16 * t) * S + q4;
                u_n[t] = a.u[f];
                l_n[t] = a.lam[f];
                if (a.grad_at_lam) g_n[t] = a.grad_at_lam[f];
            }
    };
    auto arrive = [&]() {
#pragma unroll
        for (int t = 0; t < DT; ++t) asm volatile("" : "+v"(u_n[t]), "+v"(l_n[t]), "+v"(g_n[t]));
        asm volatile("" : "+v"(dx_n), "+v"(nt_n), "+v"(tag_n));
        nt_n = __builtin_amdgcn_readfirstlane(nt_n);
        tag_n = __builtin_amdgcn_readfirstlane(tag_n);
    };
    f32x4 K[KEEP ? TILES : 1];
    auto fetch_kept = [&](long cl) {
        if constexpr (!KEEP) return;
#pragma unroll
        for (int t = 0; t < TILES; ++t) K[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (cl < 0 || tag_n != nt_n || tag_n == 0) return;
        const f32x4* src = reinterpret_cast<const f32x4*>(a.pinv + cl * wide_kept(SM)) + lane;
#pragma unroll
        for (int tr = 0; tr < NT; ++tr) {
            if (16 * tr >= S * nt_n) break;
#pragma unroll
            for (int tc = 0; tc <= tr; ++tc) K[tile_lower(tc, tr)] = src[64 * tile_lower(tc, tr)];
        }
    };
    long next = queue.first();
    prefetch(next);
    arrive();
    fetch_kept(next);
    while (next >= 0) {
        renew();
        const long cell = next;
        int nt = nt_n, n = S * nt;
        const double dx = dx_n;
        double* lg = a.lam + cell * SM;
        double* lam = wb + at.lam;
        double* lamnew = wb + at.lamnew;
        // dual (s, i) = (q4, p16 + 16 t) of the lane
        bool on[DT];
        double ue[DT], g[DT], gt[DT] = {}, d[DT] = {};
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            on[t] = q4 < S && p16 + 16 * t < nt;
            ue[t] = on[t] ? u_n[t] : 0.0;
            g[t] = on[t] ? g_n[t] : 0.0;
            if (on[t]) lam[(p16 + 16 * t) * S + q4] = l_n[t];
        }
        yb[lane] = 0.0;
        yb[64 + lane] = 0.0;
        queue.ask();
        // the kept inverse is usable where it was formed at this cell's order
        const bool reuse = KEEP && a.pinv_mode == 1 && c.max_iter != 1 && cell < a.pinv_slots;
        bool refactor = !reuse || tag_n != nt, factored = false;
        wave_sync();

        double uproj[DT] = {};
        // f(k, Lambda(k)) at the points for the duals X (LDS), two per lane at
        // a time where there are as many
        auto at_points = [&](const double* X, auto f) {
            auto part = [&](int p0, auto width) {
                constexpr int W = decltype(width)::value;
                double t4[W][4] = {};
                const double* ph[4 * W];
#pragma unroll
                for (int t = 0; t < 4 * W; ++t) {
                    const int k = p0 + 16 * t + p16;
                    ph[t] = phiT + q4 * QP + (k < Q ? k : Q - 1);
                }
                in_steps<1>(
                    (nt + 3) / 4,
                    [&](int ki) {
                        Operands<4 * W> o;
                        const int i = 4 * ki + q4;
                        o.a = i < nt ? X[i * S + s4] : 0.0;
#pragma unroll
                        for (int t = 0; t < 4 * W; ++t) o.b[t] = ph[t][4 * ki * QP];
                        return o;
                    },
                    [&](const Operands<4 * W>& o) {
#pragma unroll
                        for (int t = 0; t < 4 * W; ++t)
                            t4[t >> 2][t & 3] =
                                __builtin_amdgcn_mfma_f64_4x4x4f64(o.a, o.b[t], t4[t >> 2][t & 3], 0, 0, 0);
                    });
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    group_transpose(t4[w]);
                    double L[S];
#pragma unroll
                    for (int s = 0; s < S; ++s) L[s] = t4[w][s];
                    f(p0 + 64 * w + lane, L);
                }
            };
            int p0 = 0;
            for (; p0 + 64 < Q; p0 += 128) part(p0, std::integral_constant<int, 2>());
            if (p0 < Q) part(p0, std::integral_constant<int, 1>());
            wave_sync();
        };
        // <Ub phiW> of the lane's duals
        auto project = [&](double (&out)[DT]) {
            const double* ua = Ub + s4 * QP + 2 * q4;
            auto part = [&](auto first, auto count) {
                constexpr int t0 = decltype(first)::value, N = decltype(count)::value;
                const double* wa[N];
                double acc[N] = {};
#pragma unroll
                for (int t = 0; t < N; ++t) {
                    const int i = p16 + 16 * (t0 + t);
                    wa[t] = phiwT + (i < M ? i : M - 1) * QP + 2 * q4;
                }
                in_steps<N == 1 ? 4 : 2>(
                    QP / 8,
                    [&](int k) {
                        Operands<N, f64x2> o;
                        o.a = two(ua + 8 * k);
#pragma unroll
                        for (int t = 0; t < N; ++t) o.b[t] = two(wa[t] + 8 * k);
                        return o;
                    },
                    [&](const Operands<N, f64x2>& o) {
#pragma unroll
                        for (int h = 0; h < 2; ++h)
#pragma unroll
                            for (int t = 0; t < N; ++t)
                                acc[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(o.a[h], o.b[t][h], acc[t], 0, 0, 0);
                    });
#pragma unroll
                for (int t = 0; t < N; ++t) out[t0 + t] = acc[t];
            };
#pragma unroll
            for (int t = 0; t < DT; ++t) out[t] = 0.0;
            static_for<(DT + 1) / 2>([&](auto h) {
                constexpr int t0 = 2 * decltype(h)::value;
                if (t0 + 1 < DT && 16 * (t0 + 1) < nt) {
                    if constexpr (t0 + 1 < DT)
                        part(std::integral_constant<int, t0>(), std::integral_constant<int, 2>());
                } else if (16 * t0 < nt) {
                    part(std::integral_constant<int, t0>(), std::integral_constant<int, 1>());
                }
            });
        };
        // U at the duals X into Ub, Lambda into DUb
        auto evaluate = [&](const double* X) {
            at_points(X, [&](int k, double (&L)[S]) {
                double U[S];
                closure_U<KIND>(c, L, U);
                if (k < QP) {
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        Ub[s * QP + k] = k < Q ? U[s] : 0.0;  // (an infinity times the table's zero is NaN)
                        DUb[s * QP + k] = L[s];
                    }
                }
            });
        };
        auto norm = [&](const double (&v)[DT]) -> double {
            double sq = 0.0;
#pragma unroll
            for (int t = 0; t < DT; ++t) sq += v[t] * v[t];
            return lane_get(sqrt(wave_sum(sq)), 0);  // (in scalar registers: the branches on it are uniform)
        };
        // yb <- a vector over the duals' lanes
        auto put = [&](const double (&v)[DT]) {
#pragma unroll
            for (int t = 0; t < DT; ++t)
                if (on[t]) yb[(p16 + 16 * t) * S + q4] = v[t];
            wave_sync();
        };
        // v <- P yb, P the kept inverse: a lower tile gives the products of
        // its rows, summed over the lane groups, and of its columns, summed
        // over a group's lanes (by the diagonal tiles' full squares: once)
        auto apply_kept = [&](double (&v)[DT]) {
            // phase: matvec
            double row[NT], col[4 * NT];
#pragma unroll
            for (int r = 0; r < NT; ++r) row[r] = 0.0;
#pragma unroll
            for (int r = 0; r < 4 * NT; ++r) col[r] = 0.0;
#pragma unroll
            for (int tr = 0; tr < NT; ++tr) {
                if (16 * tr >= n) break;
                const double xr = yb[16 * tr + p16];
#pragma unroll
                for (int tc = 0; tc <= tr; ++tc)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const double k = (double)K[tile_lower(tc, tr)][e];
                        row[tr] = fma(k, yb[16 * tc + 4 * e + q4], row[tr]);
                        if (tc < tr) col[4 * tc + e] = fma(k, xr, col[4 * tc + e]);
                    }
            }
            wave_sync();
#pragma unroll
            for (int tr = 0; tr < NT; ++tr) {
                if (16 * tr >= n) break;
                const double y = group_sum(row[tr]);
                if (q4 == (tr & 3)) yb[16 * tr + p16] = y;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const double z = row_sum(col[4 * tr + e]);
                    if (p16 == (4 * tr + e) % 16) ring[16 * tr + 4 * e + q4] = z;
                }
            }
            wave_sync();
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                const int f = (p16 + 16 * t) * S + q4;
                v[t] = on[t] ? yb[f] + ring[f] : 0.0;
            }
            wave_sync();
            // phase end: matvec
        };
        // Newton direction at the iterate of the last gradient; false if the
        // Hessian is not positive definite
        auto direction = [&](const double (&g)[DT], double (&d)[DT]) -> bool {
            // phase: hessian
            // (not needed again for this cell: its registers hold the tiles)
#pragma unroll
            for (int t = 0; t < (KEEP ? TILES : 0); ++t) K[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int k = lane; k < QP - 4; k += 64) {
                double L[S], y[P];
#pragma unroll
                for (int s = 0; s < S; ++s) L[s] = DUb[s * QP + k];
                closure_DU<KIND>(c, L, Ub[k], y);  // (the last gradient was lam's)
#pragma unroll
                for (int p = 0; p < P; ++p) DUb[p * QP + k] = y[p];
            }
            put(g);
            f64x4 T[TILES];
#pragma unroll
            for (int t = 0; t < TILES; ++t) T[t] = f64x4{0.0, 0.0, 0.0, 0.0};
            const int npair = nt * (nt + 1) / 2;
            int done = 0, head = 0, first = 0;  // pairs formed; the group's first row in the ring, and packed
            // where row r of the window starts
            auto start = [&](int r) {
                const int x = ((int)__umul24(r, r + 1) >> 1) - first + head;
                return x < RS ? x : x - RS;
            };
#pragma unroll
            for (int tr = 0; tr < NT; ++tr) {
                for (int h = 0; h < 4; ++h) {
                    const int r0 = 16 * tr + 4 * h;
                    if (r0 > n) break;
                    const int il = (r0 + 3) / S < nt ? (r0 + 3) / S : nt - 1;
                    while (done < (il + 1) * (il + 2) / 2) {
                        const double *fj[2], *wi[2], *du[PG];
                        double acc[2][PG] = {};
#pragma unroll
                        for (int w = 0; w < 2; ++w) {
                            const int e = done + 16 * w + p16;
                            int j, i;
                            basis_pair(e < npair ? e : npair - 1, j, i);
                            fj[w] = phiT + j * QP + 2 * q4;
                            wi[w] = phiwT + i * QP + 2 * q4;
                        }
#pragma unroll
                        for (int pg = 0; pg < PG; ++pg) {
                            const int p = 4 * pg + (p16 & 3);
                            du[pg] = DUb + (p < P ? p : P - 1) * QP + 2 * q4;
                        }
                        struct Step {
                            f64x2 f[2], w[2], d[PG];
                        };
                        in_steps<2>(
                            QP / 8,
                            [&](int k) {
                                Step o;
#pragma unroll
                                for (int w = 0; w < 2; ++w) {
                                    o.f[w] = two(fj[w] + 8 * k);
                                    o.w[w] = two(wi[w] + 8 * k);
                                }
#pragma unroll
                                for (int pg = 0; pg < PG; ++pg) o.d[pg] = two(du[pg] + 8 * k);
                                return o;
                            },
                            [&](const Step& o) {
#pragma unroll
                                for (int h = 0; h < 2; ++h) {
                                    const double a0 = o.f[0][h] * o.w[0][h], a1 = o.f[1][h] * o.w[1][h];
#pragma unroll
                                    for (int pg = 0; pg < PG; ++pg) {
                                        acc[0][pg] =
                                            __builtin_amdgcn_mfma_f64_4x4x4f64(a0, o.d[pg][h], acc[0][pg], 0, 0, 0);
                                        acc[1][pg] =
                                            __builtin_amdgcn_mfma_f64_4x4x4f64(a1, o.d[pg][h], acc[1][pg], 0, 0, 0);
                                    }
                                }
                            });
                        // this lane's products: pair 16 w + 4 (p16 / 4) + q4, state pairs 4 pg + p16 % 4
#pragma unroll
                        for (int w = 0; w < 2; ++w) {
                            const int e = done + 16 * w + 4 * (p16 >> 2) + q4;
                            int j, i;
                            basis_pair(e < npair ? e : npair - 1, j, i);
#pragma unroll
                            for (int pg = 0; pg < PG; ++pg) {
                                const int p = 4 * pg + (p16 & 3);
                                const int l = p < 1 ? 0 : p < 3 ? 1 : p < 6 ? 2 : 3, m = p - l * (l + 1) / 2;
                                const int r1 = i * S + l, c1 = j * S + m, r2 = i * S + m, c2 = j * S + l;
                                if (e < npair && p < P) {
                                    ring[start(r1) + c1] = acc[w][pg];
                                    if (m < l && j < i) ring[start(r2) + c2] = acc[w][pg];
                                }
                            }
                        }
                        done += 32;
                    }
                    wave_sync();
                    // rows r0 .. r0 + 3, and the right-hand side as row n
                    const int r = 16 * tr + p16;
                    if ((p16 >> 2) == h && r <= n) {
                        const double* src = r < n ? ring + start(r) : yb;
#pragma unroll
                        for (int tc = 0; tc <= tr; ++tc)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const int cc = 16 * tc + 4 * e + q4;
                                if (tc < tr || cc < r || (cc == r && r < n)) T[tile_lower(tc, tr)][e] = src[cc];
                            }
                    }
                    wave_sync();
                    first += 4 * r0 + 10;
                    head += 4 * r0 + 10;
                    if (head >= RS) head -= RS;
                }
            }
            // phase end: hessian
            renew();
            asm volatile("" : "+v"(nt));
            nt = __builtin_amdgcn_readfirstlane(nt);
            n = S * nt;
            bool spd;
            if constexpr (KEEP) {
                // phase: sweep
                // the diagonal tiles' upper halves, by symmetry
#pragma unroll
                for (int tr = 0; tr < NT; ++tr) {
                    if (16 * tr >= n) break;
#pragma unroll
                    for (int e = 0; e < 4; ++e) ring[(4 * e + q4) * 17 + p16] = T[tile_lower(tr, tr)][e];
                    wave_sync();
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (4 * e + q4 > p16) T[tile_lower(tr, tr)][e] = ring[p16 * 17 + 4 * e + q4];
                    wave_sync();
                }
                spd = tile_sweep_lower<NT>(T, n, p16, q4, ring);
                // the solution in row n
#pragma unroll
                for (int tr = 0; tr < NT; ++tr)
                    if (16 * tr <= n && n < 16 * tr + 16 && p16 == (n & 15)) {
#pragma unroll
                        for (int tc = 0; tc <= tr; ++tc)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                if (16 * tc + 4 * e + q4 < n) yb[16 * tc + 4 * e + q4] = T[tile_lower(tc, tr)][e];
                    }
                if (spd && reuse) {
                    f32x4* dst = reinterpret_cast<f32x4*>(a.pinv + cell * wide_kept(SM)) + lane;
#pragma unroll
                    for (int tr = 0; tr < NT; ++tr) {
                        if (16 * tr >= n) break;
#pragma unroll
                        for (int tc = 0; tc <= tr; ++tc) {
                            f32x4 v;
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                v[e] = 16 * tr + p16 < n && 16 * tc + 4 * e + q4 < n
                                           ? (float)-T[tile_lower(tc, tr)][e]
                                           : 0.f;
                            dst[64 * tile_lower(tc, tr)] = v;
                        }
                    }
                }
                // phase end: sweep
            } else {
                // phase: factor
                spd = tile_ldl<NT>(T, n, p16, q4);
                double X[NT];
                tile_back_rows<NT>(T, n, p16, q4, X);
#pragma unroll
                for (int r = 0; r < NT; ++r)
                    if (q4 == (r & 3) && 16 * r + p16 < n) yb[16 * r + p16] = X[r];
                // phase end: factor
            }
            wave_sync();
            renew();
#pragma unroll
            for (int t = 0; t < DT; ++t) d[t] = on[t] ? yb[(p16 + 16 * t) * S + q4] : 0.0;
            wave_sync();
            return spd;
        };

        double ng = 0.0, step = 1.0;
        int status = -1, iters = 0, halvings = 0, ngrad = 0;
        bool ub_lam = false;  // Ub and uproj belong to lam
        bool asked = false;   // the next cell is sent for
        // GIVEN: the residual check left the gradient at lambda; KEPT: the
        // trial point of a step on the kept inverse; BACK: lambda again, after
        // such a step did not lower the gradient
        enum { GIVEN, START, TRIAL, KEPT, BACK, END };
        int where = a.grad_at_lam ? GIVEN : START;
        asm volatile("" : "+v"(where));  // (not cloned for its first pass)
        where = __builtin_amdgcn_readfirstlane(where);
        for (;;) {
            renew();
            asm volatile("" : "+v"(nt));
            nt = __builtin_amdgcn_readfirstlane(nt);
            n = S * nt;
#pragma unroll
            for (int t = 0; t < DT; ++t) on[t] = q4 < S && p16 + 16 * t < nt;
            // phase: gradient
            evaluate(where == TRIAL || where == KEPT ? lamnew : lam);
            double nt_norm = 0.0;
            if (where != GIVEN && where != BACK) {
                ++ngrad;
                project(uproj);
#pragma unroll
                for (int t = 0; t < DT; ++t) gt[t] = on[t] ? uproj[t] - ue[t] : 0.0;
                nt_norm = norm(gt);
            } else if (where == GIVEN) {
#pragma unroll
                for (int t = 0; t < DT; ++t) gt[t] = g[t];
                nt_norm = norm(gt);
            }
            wave_sync();
            // phase end: gradient
            if (where == END) break;
            bool full = false;  // the next step factors
            if (where == GIVEN || where == START) {
                queue.resolve();
                ng = nt_norm;
                ub_lam = where == START;
                if (!c.safe && ng < c.eps) status = UQK_STATUS_CONVERGED;
            } else if (where == KEPT) {
                ub_lam = false;
                if (nt_norm < ng) {
                    ++w_count[6];
                    double* x = lam;
                    lam = lamnew;
                    lamnew = x;
                    ub_lam = true;
                    const double ratio = nt_norm / ng;
                    ng = nt_norm;
                    // contraction clearly worse than a (damped) Newton step's:
                    // factor afresh at the next Newton step.  From n = 64 on, a
                    // factorisation (Hessian O(Q n^2), sweep O(n^3)) costs some
                    // ten steps on the kept inverse (O(n^2 + Q n)), and a step
                    // that contracts by 0.05 is still worth keeping
                    const double slack = n >= 64 ? 0.05 : 1e-3;
                    if (!(ratio <= 1.2 * (1.0 - c.alpha) + slack)) refactor = true;
                    if (nt_norm < c.eps) status = UQK_STATUS_CONVERGED;
                } else {
                    refactor = true;
                    if (iters < c.max_iter) {
                        where = BACK;
                        continue;
                    }
                }
            } else if (where == TRIAL) {
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
                if (where != BACK) {
#pragma unroll
                    for (int t = 0; t < DT; ++t) g[t] = gt[t];
                }
                full = !KEEP || !reuse || refactor;
                if (full) {
                    if (!direction(g, d)) {
                        status = UQK_STATUS_NOT_SPD;
                    } else {
                        ++w_count[5];
                        factored = reuse;
                        if (c.max_iter == 1) {  // one-shot IPM (closure.cpp:151-154)
#pragma unroll
                            for (int t = 0; t < DT; ++t)
                                if (on[t]) lam[(p16 + 16 * t) * S + q4] -= c.alpha * d[t];
                            ub_lam = false;
                            wave_sync();
                            status = UQK_STATUS_CONVERGED;
                        }
                    }
                } else if constexpr (KEEP) {
                    // d = P g + P (g - H P g): per point w(k) = DU_k (v^T
                    // phi_k), then H v = <w phiW> -- the Hessian of
                    // closure.cpp:255-271 applied to v = P g, in place of U
                    double d1[DT], hv[DT];
                    put(g);
                    apply_kept(d1);
#pragma unroll
                    for (int t = 0; t < DT; ++t)
                        if (on[t]) lamnew[(p16 + 16 * t) * S + q4] = d1[t];
                    wave_sync();
                    // phase: hessvec
                    at_points(lamnew, [&](int k, double (&L)[S]) {
                        if (k < QP) {
                            double Lk[S], y[P];
#pragma unroll
                            for (int s = 0; s < S; ++s) Lk[s] = DUb[s * QP + k];
                            closure_DU<KIND>(c, Lk, Ub[k], y);
#pragma unroll
                            for (int l = 0; l < S; ++l) {
                                double w = 0.0;
#pragma unroll
                                for (int m = 0; m < S; ++m)
                                    w += y[l >= m ? l * (l + 1) / 2 + m : m * (m + 1) / 2 + l] * L[m];
                                Ub[l * QP + k] = k < Q ? w : 0.0;
                            }
                        }
                    });
                    project(hv);
#pragma unroll
                    for (int t = 0; t < DT; ++t) hv[t] = on[t] ? g[t] - hv[t] : 0.0;
                    // phase end: hessvec
                    put(hv);
                    apply_kept(d);
#pragma unroll
                    for (int t = 0; t < DT; ++t) d[t] += d1[t];
                    ub_lam = false;
                }
            }
            if (!asked) {
                asked = true;
                next = queue.take();
                prefetch(next);
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
                where = full ? TRIAL : KEPT;
                continue;
            }
            // the outputs come from U at the returned lambda
            if (!a.uq_out || ub_lam) break;
            where = END;
        }
        // phase: outputs
        arrive();
        fetch_kept(next);
        // the slot for the next steps: this call's last inverse; none after a
        // step on the kept one did poorly
        if (reuse && lane == 0) {
            const bool keep = factored && status != UQK_STATUS_NOT_SPD;
            if (keep || refactor) a.pinv_ok[cell] = keep ? nt : 0;
        }
        for (int t = lane; t < n; t += 64) lg[t] = lam[t];
        if (a.uq_out) {
            // the step's next two sweeps from the gradient at the returned
            // lambda: uQ = U(lambda phi) (momentsolver.cpp:100) and u = <uQ
            // phiW> over the cell's nTotal, zero above (:120-124)
            double* uqg = a.uq_out + cell * (long)Q * S;
            for (int t = lane; t < Q * S; t += 64) {
                const int k = t / S, s = t - k * S;
                uqg[t] = Ub[s * QP + k];
            }
#pragma unroll
            for (int t = 0; t < DT; ++t)
                if (q4 < S && p16 + 16 * t < M)
                    a.u_out[cell * SM + (p16 + 16 * t) * S + q4] = on[t] ? uproj[t] : 0.0;
            if (a.dt_min) {  // momentsolver.cpp:127-133 for this cell
                double m = 1e10;
                for (int k = lane; k < Q; k += 64) {
                    double uk[S];
#pragma unroll
                    for (int s = 0; s < S; ++s) uk[s] = Ub[s * QP + k];
                    m = fmin(m, point_dt<S>(a.dtp, uk, dx));
                }
                const double mc = wave_min(m);
                w_dt = fmin(w_dt, mc);
                if (a.dt_cell && lane == 0) a.dt_cell[cell] = mc;
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

// wavefronts per workgroup: one per SIMD, fewer where the LDS holds no more
inline int wide_waves(int S, int M, int Q, int max_lds, size_t* bytes = nullptr) {
    const WideLds at(S, M, Q, wide_ring(S, M));
    for (int w = 4; w > 0; --w) {
        const size_t b = sizeof(double) * ((size_t)at.tables + (size_t)w * at.wave);
        if (bytes) *bytes = b;
        if (b <= (size_t)max_lds) return w;
    }
    return 0;
}

template <int KIND, int NT, bool KEEP>
static hipError_t wide_go(const NewtonArgs& args, int max_lds, int num_cu, hipStream_t st, const LaunchShape& shape) {
    constexpr int S = KindInfo<KIND>::S;
    NewtonArgs a = args;
    a.wave_doubles = wide_ring(S, a.M);
    const WideLds at(S, a.M, a.Q, a.wave_doubles);
    const int waves = wide_waves(S, a.M, a.Q, max_lds);  // (shape.waves is the wave kernel's)
    if (waves < 1) return hipErrorInvalidValue;
    const size_t shmem = sizeof(double) * ((size_t)at.tables + (size_t)waves * at.wave);
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, newton_wide_kernel<KIND, NT, KEEP>, 64 * waves, shmem) !=
            hipSuccess ||
        occ <= 0)
        occ = 1;
    if (shape.blocks_per_cu > 0 && shape.blocks_per_cu < occ) occ = shape.blocks_per_cu;
    const long want = a.ncell, cap = (long)occ * (num_cu > 0 ? num_cu : 1);
    const unsigned blocks = (unsigned)(want < cap ? (want > 0 ? want : 1) : cap);
    hipLaunchKernelGGL((newton_wide_kernel<KIND, NT, KEEP>), dim3(blocks), dim3(64 * waves), shmem, st, a);
    return hipGetLastError();
}

template <int KIND>
static hipError_t wide_kind(const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st, const LaunchShape& shape) {
    const bool keep = a.pinv_mode == 1 && a.c.max_iter != 1;
    switch (wide_tiles(KindInfo<KIND>::S * a.M)) {
        case 1: case 2: case 3: case 4: case 5:
        case 6: return (keep ? wide_go<KIND, 6, true> : wide_go<KIND, 6, false>)(a, max_lds, num_cu, st, shape);
        case 7: return (keep ? wide_go<KIND, 7, true> : wide_go<KIND, 7, false>)(a, max_lds, num_cu, st, shape);
        case 8:
            if constexpr (wide_limit(KindInfo<KIND>::S) > 111)
                return (keep ? wide_go<KIND, 8, true> : wide_go<KIND, 8, false>)(a, max_lds, num_cu, st, shape);
    }
    return hipErrorInvalidValue;
}

}  // namespace uqk
