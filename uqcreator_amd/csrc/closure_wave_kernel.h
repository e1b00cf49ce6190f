// closure_wave_kernel.h -- the one-wavefront Newton closure kernel template
// and its launch helpers, shared by closure_wave.hip (FP64 and mixed
// instantiations, the dispatch), closure_wave_reuse.hip (the mixed closure
// with the reuse of the factorisation across time steps) and
// closure_wave_lag.hip (the same within one closure call).
//
// Batched Newton dual closure, one wavefront per cell, specialised at compile
// time for the (closure, M, Q) of a config with n = S*M <= 63 duals, M <= 16
// and Q <= 64 quadrature points.  Same algorithm as closure_fp64.hip
// (Closure::SolveClosure / SolveClosureSafe, closure.cpp:133-193, :297-339),
// laid out for wave64 and its FP64 matrix instructions:
//   * lane k owns quadrature point k: it evaluates Lambda(k) = lambda^T phi(k),
//     U and DU there;
//   * lane 16 s + i owns dual (s, i) of the moments, gradient, trial gradient
//     and Newton direction -- the output layout of v_mfma_f64_4x4x4_4b, so
//     the projection <U phiW> (one such product per four points) needs no
//     transposition and the line search runs in registers;
//   * Hessian (closure.cpp:255-271): H_(s,i)(t,j) = sum_k phi_i phiW_j DU_st
//     depends on the basis pair (j <= i) and the state pair only, so it is the
//     product (pairs x points)(points x state pairs) on v_mfma_f64_4x4x4_4b,
//     75-83% of whose slots are used (16 x 16 blocks per state pair: 39% at
//     M = 10).  The pair products go to LDS and from there, by a table of
//     addresses, into the tiles of tile_solve.h;
//   * factorisation (dposv 'U', vectorspace.cpp:152-171) and solve, or the
//     explicit inverse where steps reuse it, in registers: tile_solve.h.
//
// What bounds it: the latency of one cell's chain of dependent steps at two
// wavefronts per SIMD, most of it instruction issue.  Cycles per call at n =
// 40, 25 points (Euler 2D, FP64): factorisation 13.1 K and back substitution
// 3.4 K (register tiles spread over the wave with one LDS round trip per two
// pivots: 23.4 K and 19.2 K), Hessian 3.7 K (pairs over lanes, DU by
// v_readlane, with an exponential and a logarithm: 14.6 K), gradient 3.6 K
// (4.3 K); 65,536 cells, 40 time steps: 20.2 ms against 39.0 (FP64), 15.4
// against 30.7 (mixed).  At n = 45, 49 points, one closure of 100,003 cells:
// 29.2 ms against 47.4 (FP64), 10.0 against 19.5 (mixed: a step on the kept
// inverse is a matrix-vector product from registers, 1.3 K cycles, in place
// of two triangular solves from LDS, 13.9 K).
// The next cell's moments, duals, density and kept inverse are asked for
// while this cell still computes and are waited for before its results are
// stored: loads come back in order behind the stores that precede them, and
// asked for at the cell's end they cost 2.1 ms more over the mixed loop above.
#pragma once
#include <hip/hip_runtime.h>

#include "cell_queue.h"
#include "tile_solve.h"
#include "uqk_device.h"
#include "uqk_internal.h"

namespace uqk {

template <int KIND, int M, int Q>
struct WaveShape {
    static constexpr int S = KindInfo<KIND>::S;
    static constexpr int N = S * M;              // duals per cell
    static constexpr int P = S * (S + 1) / 2;    // distinct DU entries
    static constexpr int KS = (Q + 3) / 4;       // four points per matrix step
    // row length of the tables and of U: 4 mod 8, as tile_solve.h's f64x2 reads like it
    static constexpr int QP = 4 * KS + (KS % 2 ? 0 : 4);
    // the point that lane group q has in step ks: two steps share eight points,
    // of which a group takes two neighbours (one read); a last odd step has four
    __host__ __device__ static constexpr int point(int ks, int q) {
        return (ks | 1) < KS ? 8 * (ks / 2) + 2 * q + (ks & 1) : 4 * ks + q;
    }
    static constexpr int NPAIR = M * (M + 1) / 2;
    static constexpr int PT = (NPAIR + 15) / 16; // tiles of 16 basis pairs
    static constexpr int PG = (P + 3) / 4;       // groups of four state pairs
    static constexpr int NT = N / 16 + 1;        // 16-row tiles of the system and its right-hand side
    // per-wave LDS doubles
    static constexpr int LAM = 0;
    static constexpr int LAMNEW = LAM + N;
    static constexpr int UB = (LAMNEW + N + 1) & ~1;  // U values, S rows of QP
    static constexpr int YB = UB + S * QP;            // 64: a vector over the unknowns
    // pair products (4 PG rows of NPAIR), the right-hand side (N), zero (1);
    // before them, in the same place, DU at the points (P rows of QP)
    static constexpr int BH = YB + 64;
    static constexpr int BH_RHS = 4 * PG * NPAIR;
    static constexpr int BH_ZERO = BH_RHS + N;
    static constexpr int BH_SIZE = BH_ZERO + 1 > P * QP ? BH_ZERO + 1 : P * QP;
    static constexpr int WAVE_DOUBLES = (BH + BH_SIZE + 1) & ~1;
    // tables of the workgroup: phi and phiw (i-major), the products phi_i
    // phiw_j of the pairs in operand order where they take at most 16 KB
    // (else they are formed from the two tables), the tile addresses
    static constexpr bool PAIR_TABLE = PT * KS * 64 * 8 <= 16384;
    static constexpr int KI = (M + 3) / 4;       // four basis functions per matrix step
    static constexpr int QT = (Q + 15) / 16;     // tiles of 16 points
    static constexpr int PHIW = 4 * KI * QP;     // phi: rows padded with zero to 4 KI
    static constexpr int PAIRS = PHIW + M * QP;
    static constexpr int ADDR = PAIRS + (PAIR_TABLE ? PT * KS * 64 : 0);
    // kept inverse (PREC 2): row r's entries 4 t + q of lane group q in a run
    static constexpr int NQ = (N + 3) / 4;
    static constexpr int KEPT = 4 * NQ * N;
};

// PREC 0: FP64, and the mixed path where nothing is reused (a one-shot or
// undamped closure call).  PREC 2: the reuse of the factorisation across time
// steps (the time loop's mixed closure).  PREC 4: the reuse within one closure
// call (a cell's later Newton steps apply its last inverse while they
// contract).
template <int PREC> constexpr bool wave_reuses = PREC == 2 || PREC == 4;

// tile registers of the system: all of it where later steps of the call apply
// the inverse from the registers, the lower triangle otherwise
template <int PREC, int NT> constexpr int wave_tiles = PREC == 4 ? NT * NT : NT * (NT + 1) / 2;

__device__ __forceinline__ f64x2 two(const __attribute__((address_space(3))) double* x) {
    return *reinterpret_cast<const __attribute__((address_space(3))) f64x2*>(x);
}
// a row of LDS (of points) as the operands of all KS steps: WaveShape::point
template <int KS, class D>
__device__ __forceinline__ void row_steps(const D* row, int q4, double (&v)[KS]) {
#pragma unroll
    for (int ks = 0; ks + 1 < KS; ks += 2) {
        const f64x2 x = two(row + 4 * ks + 2 * q4);
        v[ks] = x[0];
        v[ks + 1] = x[1];
    }
    if constexpr (KS % 2) v[KS - 1] = row[4 * (KS - 1) + q4];
}

// The system of a Newton step at the iterate whose Lambda and density lie at
// this lane's point in Lk and rk, into bh: the pair products (pairs x points)(points x state
// pairs) on FP64 matrix steps; with RHS also the gradient g of this lane's
// dual (the right-hand side).  smem: the workgroup's tables, bh: the wave's.
template <int KIND, int M, int Q, bool RHS, class D>
__device__ __forceinline__ void wave_system(const ClosureParams& c, const double* Lk, double rk, double g, D* smem,
                                            D* bh, int lane, int p16, int q4) {
    using W = WaveShape<KIND, M, Q>;
    constexpr int S = W::S, P = W::P, QP = W::QP, KS = W::KS;
    double y[P];
    closure_DU<KIND>(c, Lk, rk, y);
    if (lane < QP) {
#pragma unroll
        for (int p = 0; p < P; ++p) bh[p * QP + lane] = y[p];
    }
    wave_sync();
    double du[W::PG][KS];
#pragma unroll
    for (int pg = 0; pg < W::PG; ++pg) {
        const int p = 4 * pg + (p16 & 3);
        row_steps<KS>(bh + (p < P ? p : P - 1) * QP, q4, du[pg]);
    }
    wave_sync();
    // products of tile t: lane holds (pair 16 t + 4 (p16 / 4) + q4, state pair 4 pg + p16 % 4)
    D* out = bh + (p16 & 3) * W::NPAIR + 4 * (p16 >> 2) + q4;
#pragma unroll
    for (int t = 0; t < W::PT; ++t) {
        double acc[W::PG];
#pragma unroll
        for (int pg = 0; pg < W::PG; ++pg) acc[pg] = 0.0;
        double fj[KS], wi[KS];
        if constexpr (!W::PAIR_TABLE) {
            int j, i;
            basis_pair(16 * t + p16 < W::NPAIR ? 16 * t + p16 : 0, j, i);
            row_steps<KS>(smem + j * QP, q4, fj);
            row_steps<KS>(smem + W::PHIW + i * QP, q4, wi);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            double av;
            if constexpr (W::PAIR_TABLE)
                av = smem[W::PAIRS + (t * KS + ks) * 64 + lane];
            else
                av = fj[ks] * wi[ks];
#pragma unroll
            for (int pg = 0; pg < W::PG; ++pg)
                acc[pg] = __builtin_amdgcn_mfma_f64_4x4x4f64(av, du[pg][ks], acc[pg], 0, 0, 0);
        }
        if (16 * t + 15 < W::NPAIR || 16 * t + 4 * (p16 >> 2) + q4 < W::NPAIR) {
#pragma unroll
            for (int pg = 0; pg < W::PG; ++pg) out[4 * pg * W::NPAIR + 16 * t] = acc[pg];
        }
    }
    if constexpr (RHS) {
        if (q4 < S && p16 < M) bh[W::BH_RHS + q4 * M + p16] = g;
    }
    if (lane == 0) bh[W::BH_ZERO] = 0.0;
    wave_sync();
}

// A factored step of the reuse across time steps (PREC 2): forms the system,
// sweeps it, leaves H^-1 g in yb (by unknown) and, where Pg is given, --
// rounded to FP32 -- H^-1 in the cell's slot.  A function of its own, not
// inlined: in the time loop one step in six factors, and inlined its registers
// made the other steps' inputs spill (every reload then waits for the stores
// before it).  smem: the workgroup's tables, wb: the wave's LDS.
typedef __attribute__((address_space(3))) double lds_double;
typedef __attribute__((address_space(3))) unsigned lds_unsigned;
template <int KIND, int M, int Q>
__device__ __attribute__((noinline)) bool sweep_step(ClosureParams c, double L0, double L1, double L2, double L3,
                                                     double rk, double g, lds_double* smem, lds_double* wb, float* Pg) {
    using W = WaveShape<KIND, M, Q>;
    constexpr int N = W::N, NT = W::NT, TILES = NT * (NT + 1) / 2, NQ = W::NQ;
    const int lane = threadIdx.x & 63, p16 = lane & 15, q4 = lane >> 4;
    lds_double *bh = wb + W::BH, *yb = wb + W::YB;
    const lds_unsigned* addr = (lds_unsigned*)(smem + W::ADDR);
    const double Lk[4] = {L0, L1, L2, L3};
    wave_system<KIND, M, Q, true>(c, Lk, rk, g, smem, bh, lane, p16, q4);
    f64x4 T[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const unsigned w0 = addr[t * 128 + lane], w1 = addr[t * 128 + 64 + lane];
        T[t] = f64x4{bh[w0 & 0xffff], bh[w0 >> 16], bh[w1 & 0xffff], bh[w1 >> 16]};
    }
    const bool spd = tile_sweep_lower<NT>(T, N, p16, q4, bh);
    if (p16 == N % 16) {  // row N of the swept system
#pragma unroll
        for (int t = 0; t < NQ; ++t) yb[4 * t + q4] = T[tile_lower(t >> 2, N / 16)][t & 3];
    }
    wave_sync();
    if (spd && Pg) {
        // (r, c) of the lower tiles to both of its places, and zero to the
        // places past N that fill a row's runs (later steps read whole runs)
#pragma unroll
        for (int r = 0; r < NT; ++r)
#pragma unroll
            for (int cc = 0; cc <= r; ++cc)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int R = 16 * r + p16, C = 16 * cc + 4 * e + q4;
                    const float v = R < N && C < N ? -(float)T[tile_lower(cc, r)][e] : 0.f;
                    if (R < N && C < 4 * NQ) Pg[(R * 4 + q4) * NQ + 4 * cc + e] = v;
                    if (cc < r && C < N && R < 4 * NQ) Pg[(C * 4 + (p16 & 3)) * NQ + 4 * r + (p16 >> 2)] = v;
                }
    }
    return spd;
}

template <int KIND, int M, int Q, int PREC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) newton_wave_kernel(NewtonArgs a) {
    using W = WaveShape<KIND, M, Q>;
    constexpr int S = W::S, N = W::N, P = W::P, QP = W::QP, KS = W::KS, NT = W::NT;
    constexpr int TILES = wave_tiles<PREC, NT>;
    static_assert(N < 64 && Q <= 64, "wave kernel needs n < 64 and Q <= 64");
    static_assert(M <= 16 && S <= 4, "the projection takes one 4 x 16 tile");
    extern __shared__ double smem[];
    // (both loads are sent before either is looked at)
    const int active = a.active ? *a.active : 1;
    const long ncells = a.cell_list ? (long)*a.cell_count : a.ncell;
    if (!active || (long)blockIdx.x >= ncells) return;  // no cell for any wavefront of this workgroup
    int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    int p16 = lane & 15, q4 = lane >> 4;
    double* phiT = smem;              // phiT[i*QP + k]  = phi(k, i), zero past Q
    double* phiwT = smem + W::PHIW;   // phiwT[i*QP + k] = phiw(k, i)
    for (int t = threadIdx.x; t < W::PHIW; t += blockDim.x) {
        const int i = t / QP, k = t - i * QP;
        const bool in = k < Q && i < M;
        phiT[t] = in ? a.phi[k * M + i] : 0.0;
        if (i < M) phiwT[t] = in ? a.phiw[k * M + i] : 0.0;
    }
    double* pairs = smem + W::PAIRS;
    if constexpr (W::PAIR_TABLE) {
        // operand (pair 16 t + l % 16, point(ks, l / 16)) at (t KS + ks) 64 + l
        for (int t = threadIdx.x; t < W::PT * KS * 64; t += blockDim.x) {
            const int ln = t & 63, ks = (t >> 6) % KS, e = 16 * ((t >> 6) / KS) + (ln & 15), k = W::point(ks, ln >> 4);
            int j, i;
            basis_pair(e < W::NPAIR ? e : 0, j, i);
            pairs[t] = k < Q ? a.phi[k * M + j] * a.phiw[k * M + i] : 0.0;
        }
    }
    // address in BH of element (r = 16 tr + l % 16, c = 16 tc + 4 e + l / 16)
    // of the system, two elements (e, e + 1) to a word
    unsigned* addr = reinterpret_cast<unsigned*>(smem + W::ADDR);
    for (int t = threadIdx.x; t < TILES * 128; t += blockDim.x) {
        const int ln = t & 63, half = (t >> 6) & 1, tile = t >> 7;
        int tr, tc;
        if constexpr (PREC == 4) {
            tr = tile / NT;
            tc = tile % NT;
        } else {
            basis_pair(tile, tc, tr);
        }
        unsigned word = 0;
        for (int h = 0; h < 2; ++h) {
            const int r = 16 * tr + (ln & 15), c = 16 * tc + 4 * (2 * half + h) + (ln >> 4);
            const int hi = r > c ? r : c, lo = r > c ? c : r;
            int at = W::BH_ZERO;
            if (hi < N) {
                const int l = hi / M, m = lo / M, x = hi - l * M, y = lo - m * M;
                const int i = x > y ? x : y, j = x > y ? y : x;
                at = (l * (l + 1) / 2 + m) * W::NPAIR + i * (i + 1) / 2 + j;
            } else if (hi == N && lo < N && PREC != 4) {
                at = W::BH_RHS + lo;
            }
            word |= (unsigned)at << (16 * h);
        }
        addr[t] = word;
    }
    __syncthreads();
    double* wb = smem + W::ADDR + TILES * 64 + wave * W::WAVE_DOUBLES;
    double* lamA = wb + W::LAM;
    double* lamB = wb + W::LAMNEW;
    double* Ub = wb + W::UB;
    double* yb = wb + W::YB;
    double* bh = wb + W::BH;
    // the places past Q stay zero: an infinite U would give NaN there, against
    // the table's zero, and the line search has to see the infinity
    for (int t = lane; t < S * (QP - Q); t += 64) Ub[t % S * QP + Q + t / S] = 0.0;

    // this lane's dual (s, i) = (q4, p16): its place in a cell's arrays and
    // its unknown in the system
    bool on = q4 < S && p16 < M;
    int dj = on ? p16 * S + q4 : 0, de = on ? q4 * M + p16 : 0;
    // the lane's coordinates anew: the masks and LDS addresses that derive
    // from them are then formed where they are used instead of being kept in
    // registers over a loop
    auto renew = [&]() {
        asm volatile("" : "+v"(lane));
        p16 = lane & 15;
        q4 = lane >> 4;
        on = q4 < S && p16 < M;
        dj = on ? p16 * S + q4 : 0;
        de = on ? q4 * M + p16 : 0;
    };
    const ClosureParams& c = a.c;
    const int SM = S * M;

    // The wavefront's cells (cell_queue.h): all of them, or the ones that the
    // residual check listed.  The next cell is sent for while the current
    // one starts, and its moments, duals and flags are loaded before the
    // current cell's results are stored, so neither latency stands between
    // cells.  Wavefront w of workgroup b is worker w gridDim + b: few cells
    // go to as many workgroups.
    unsigned long long w_count[7] = {};  // as the launch's counters
    double w_dt = 1e10;                  // min ComputeDt over this wave's cells (fused path)
    CellQueue queue((long)wave * gridDim.x + blockIdx.x, (long)gridDim.x * (blockDim.x >> 6), ncells, a.cell_list,
                    a.counter);
    // a cell's inputs, loaded ahead (a lane's dual of the moments, the duals,
    // the learned start and the residual check's gradient); the kept-inverse
    // flag and the ComputeDt length are wave-uniform.  The kept inverse
    // itself is loaded ahead too: its registers are free once a cell's last
    // step is taken.
    // They are sent for once the cell's first direction is known; the reuse
    // across time steps has no registers for them then, and sends for them at
    // the cell's end.
    constexpr bool kEarly = PREC != 2;
    // (with the check's gradient also the density at the point, of the uQ that
    // the check or the last step left at lambda)
    constexpr bool kDensity = KIND == UQK_EULER1D || KIND == UQK_EULER2D;
    double u_n = 0.0, l_n = 0.0, la_n = 0.0, dx_n = 0.0, g_n = 0.0, rk_n = 0.0;
    int kf_n = 0;
    auto prefetch = [&](long cl) {
        if (cl < 0) return;
        if (on) {
            u_n = a.u[cl * SM + dj];
            l_n = a.lam[cl * SM + dj];
            if (a.lam_alt) la_n = a.lam_alt[cl * SM + dj];
            if (a.grad_at_lam) g_n = a.grad_at_lam[cl * SM + dj];
        }
        if (kDensity && a.grad_at_lam) rk_n = a.uq_out[(cl * Q + (lane < Q ? lane : Q - 1)) * S];
        if (a.uq_out && a.dt_min) dx_n = a.dx_param[cl];
        if constexpr (PREC == 2) kf_n = (a.pinv_mode == 1 && cl < a.pinv_slots) ? a.pinv_ok[cl] : 0;
    };
    constexpr int KT = PREC == 2 ? NT : 1, KQ = PREC == 2 ? W::NQ : 1;
    // waits for the inputs: what is stored next is then not waited for with
    // them (loads and stores are counted in one order)
    auto arrive = [&]() {
        asm volatile("" : "+v"(u_n), "+v"(l_n), "+v"(la_n), "+v"(g_n), "+v"(rk_n), "+v"(dx_n), "+v"(kf_n));
        kf_n = __builtin_amdgcn_readfirstlane(kf_n);
    };
    long next = queue.first();
    prefetch(next);
    arrive();
    while (next >= 0) {
        const long cell = next;

        const double la_c = la_n, dx_c = dx_n, g_c = g_n, rk_c = rk_n;
        const int kf_c = kf_n;
        // the kept inverse, sent for before Lambda at the points is formed
        // (lanes past row N - 1 repeat it; their sums are not used)
        float kept[KT][KQ];
        if constexpr (PREC == 2) {
#pragma unroll
            for (int r = 0; r < KT; ++r)
#pragma unroll
                for (int t = 0; t < KQ; ++t) kept[r][t] = 0.f;
            if (kf_c == 1) {
#pragma unroll
                for (int r = 0; r < KT; ++r) {
                    const int row = 16 * r + p16 < N ? 16 * r + p16 : N - 1;
                    const float* src = a.pinv + cell * (long)W::KEPT + (row * 4 + q4) * W::NQ;
#pragma unroll
                    for (int t = 0; t < KQ; ++t) kept[r][t] = src[t];
                }
            }
        }
        const double ue = on ? u_n : 0.0;
        double* lg = a.lam + cell * SM;
        if (on) lamA[dj] = l_n;
        queue.ask();
        wave_sync();

        double Lk[S], rk = rk_c;  // Lambda and density at this lane's point for the last gradient
        double uproj = 0.0;  // <U phiW> of this lane's dual at the last gradient
        // sum_k Ub(s, k) phiW(k, i) for this lane's dual (s, i): the product
        // (S x Q)(Q x M) in steps of four points; its lane layout is the duals'
        auto project_ub = [&]() -> double {
            // (points in order: the residual check's sum to the last bit)
            const double* ua = Ub + ((p16 & 3) < S ? (p16 & 3) : S - 1) * QP + q4;
            const double* wa = phiwT + (p16 < M ? p16 : M - 1) * QP + q4;
            double acc = 0.0;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                acc = __builtin_amdgcn_mfma_f64_4x4x4f64(ua[4 * ks], wa[4 * ks], acc, 0, 0, 0);
            return acc;
        };
        // Lambda at this lane's point (lanes past Q repeat the last one) for
        // the duals X (LDS, a cell's layout): the product (S x M)(M x points)
        // in steps of four basis functions; lane group s holds state s of 16
        // points per tile, and the tiles and groups are then exchanged
        auto point_lambda = [&](const double* X, double* L) {
            double t4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int ki = 0; ki < W::KI; ++ki) {
                const int i = 4 * ki + q4;
                const double xa = X[(i < M ? i : M - 1) * S + ((p16 & 3) < S ? (p16 & 3) : S - 1)];
#pragma unroll
                for (int t = 0; t < W::QT; ++t) {
                    const int k = 16 * t + p16;
                    t4[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(xa, phiT[i * QP + (k < Q ? k : Q - 1)], t4[t], 0, 0, 0);
                }
            }
            if constexpr (W::QT < 4) {
                // lanes past the last tile: its values again (finite)
#pragma unroll
                for (int t = W::QT; t < 4; ++t) t4[t] = t4[W::QT - 1];
            }
            group_transpose(t4);
#pragma unroll
            for (int s = 0; s < S; ++s) L[s] = t4[s];
        };
        // gradient at X (LDS); returns ||g||, leaves g_e in gout, Lambda in Lk
        auto gradient = [&](const double* X, double& gout) -> double {
            // phase: gradient
            double L[S], Uv[S];
            point_lambda(X, L);
            closure_U<KIND>(c, L, Uv);
            if (lane < Q) {
#pragma unroll
                for (int s = 0; s < S; ++s) Ub[s * QP + lane] = Uv[s];
            }
#pragma unroll
            for (int s = 0; s < S; ++s) Lk[s] = L[s];
            rk = Uv[0];
            wave_sync();
            const double acc = project_ub();
            uproj = acc;
            const double g = on ? acc - ue : 0.0;
            gout = g;
            const double nrm = sqrt(wave_sum(g * g));
            wave_sync();
            // phase end: gradient
            return nrm;
        };

        auto load_system = [&](f64x4 (&T)[TILES]) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                const unsigned w0 = addr[t * 128 + lane], w1 = addr[t * 128 + 64 + lane];
                T[t] = f64x4{bh[w0 & 0xffff], bh[w0 >> 16], bh[w1 & 0xffff], bh[w1 >> 16]};
            }
            wave_sync();
        };

        // a vector held by unknown (lane l: entry l) to the duals' lanes
        auto to_duals = [&](double v) -> double {
            yb[lane] = v;
            wave_sync();
            const double r = yb[de];
            wave_sync();
            return on ? r : 0.0;
        };
        // x_{16 r + p16}, r < NT, in every lane group -> the duals' lanes
        auto rows_to_duals = [&](const double* X) -> double {
            double v = X[0];
#pragma unroll
            for (int r = 1; r < NT; ++r) v = q4 == r ? X[r] : v;
            return to_duals(v);
        };
        // this lane group's entries 4 t + q4 of a vector over the duals' lanes
        auto columns_of = [&](double v, double (&vc)[W::NQ]) {
            if (on) yb[de] = v;
            if (N % 4 && lane >= N && lane < 4 * W::NQ) yb[lane] = 0.0;
            wave_sync();
#pragma unroll
            for (int t = 0; t < W::NQ; ++t) vc[t] = yb[4 * t + q4];
            wave_sync();
        };
        // H^-1 v with the inverse (negated) that the sweep left in T (PREC 4)
        auto apply_inverse = [&](const f64x4 (&T)[PREC == 4 ? TILES : 1], double v) -> double {
            // phase: matvec
            double vc[W::NQ], X[NT];
            columns_of(v, vc);
#pragma unroll
            for (int r = 0; r < NT; ++r) {
                double s = 0.0;
#pragma unroll
                for (int t = 0; t < W::NQ; ++t) s = fma(-T[r * NT + (t >> 2)][t & 3], vc[t], s);
                X[r] = group_sum(s);
            }
            const double d = rows_to_duals(X);
            // phase end: matvec
            return d;
        };

        // ---- reuse of the factorisation (mixed precision) ----------------
        // The kept approximation of the inverse Hessian is P = H^-1 of an
        // earlier step, rounded once to FP32, in the registers `kept`: entry
        // (16 r + p16, 4 t + q4) in kept[r][t].  FP64 accumulation.
        auto pmatvec = [&](double v) -> double {
            // phase: matvec
            double vc[W::NQ], X[NT];
            columns_of(v, vc);
#pragma unroll
            for (int r = 0; r < KT; ++r) {
                double s = 0.0;
#pragma unroll
                for (int t = 0; t < KQ; ++t) s = fma((double)kept[r][t], vc[t], s);
                X[r] = group_sum(s);
            }
            const double d = rows_to_duals(X);
            // phase end: matvec
            return d;
        };
        // (H v)_e of the FP64 Hessian at the iterate of the last gradient
        // (Lambda in Lk), without forming H: per point k, w = DU_k (v^T phi_k),
        // then sum_k w_s(k) phiW(k, i) -- the Hessian of closure.cpp:255-271
        // applied to v.  Overwrites Ub (the next gradient rewrites it).
        auto hessvec = [&](double v) -> double {
            // phase: hessvec
            if (on) yb[dj] = v;
            wave_sync();
            double Ld[S];
            point_lambda(yb, Ld);  // v^T phi_k
            double y[P];
            closure_DU<KIND>(c, Lk, rk, y);
            wave_sync();
            if (lane < Q) {
#pragma unroll
                for (int l = 0; l < S; ++l) {
                    double w = 0.0;
#pragma unroll
                    for (int m = 0; m < S; ++m) w += y[l >= m ? l * (l + 1) / 2 + m : m * (m + 1) / 2 + l] * Ld[m];
                    Ub[l * QP + lane] = w;
                }
            }
            wave_sync();
            const double hv = project_ub();
            wave_sync();
            // phase end: hessvec
            return on ? hv : 0.0;
        };

        double* lam = lamA;
        double* lamnew = lamB;
        double g = 0.0, ng = 0.0, d = 0.0, step = 1.0;
        // reuse of the factorisation (mixed precision): the cell's kept
        // inverse P is usable when pinv_ok[cell] == 1; a factored step stores
        // its own.  PREC 4 (one closure call): the inverse of this cell's last
        // Hessian stays in registers, and the next steps apply it (lagged
        // steps) until one contracts poorly or is rejected.
        bool reuse = false, refactor = true, factored = false, lagged = false;
        if constexpr (PREC == 2) {
            if (a.pinv_mode == 1 && c.max_iter != 1 && cell < a.pinv_slots) {
                reuse = true;
                refactor = kf_c != 1;
            }
        }
        if constexpr (PREC == 4) reuse = c.max_iter != 1;
        f64x4 T_call[PREC == 4 ? TILES : 1];  // (kept across the call's steps)
        double Lk0[S], rk0 = 0.0, g0 = 0.0;  // Lambda, density and gradient at lam while another point is tried
        int status = -1, iters = 0, halvings = 0;
        int ngrad = 0;  // gradients evaluated here (the residual check counts the one it gives)
        // Ub and uproj hold U and <U phiW> at lam, the outputs' source
        bool ub_lam = false;
        // The gradient is evaluated in one place, at the cell's start, at the
        // learned start, at a trial point of the line search or, for the
        // outputs, at the end; what follows depends on which it was.
        enum { GIVEN, START, ALT, TRIAL, END };
        int where = START;
        double* at = lam;
        if (a.grad_at_lam) {
            // the residual check's gradient at lambda (its projection summed in
            // point order); Lambda at this lane's point for the first Hessian
            // phase: start
            point_lambda(lam, Lk);
            g = on ? g_c : 0.0;
            ng = sqrt(wave_sum(g * g));
            where = GIVEN;
            // phase end: start
        }
        // (opaque, so that the loop is not cloned for its first pass)
        int resolved = 0;
        asm volatile("" : "+s"(where), "+s"(resolved));
        for (;;) {
            renew();
            double gt = 0.0, nt = 0.0;
            if (where != GIVEN) {
                ++ngrad;
                nt = gradient(at, gt);
            }
            if (!resolved) {
                queue.resolve();
                resolved = 1;
            }
            if (where == END) break;
            if (where == TRIAL) {
                // line search (closure.cpp:159-184): halve the step until
                // ||grad|| does not grow (SolveClosureSafe: and is finite)
                ub_lam = false;
                if (halvings > 0 && nt < c.eps) {
                    status = UQK_STATUS_CONVERGED;
                } else if (halvings > 0 && halvings > c.max_halvings) {
                    status = UQK_STATUS_LINE_SEARCH;
                } else if (!lagged && (ng < nt || (c.safe && !isfinite(nt)))) {
                    step *= 0.5;
                    ++halvings;
                    if (on) lamnew[dj] = lam[dj] - step * c.alpha * d;
                    wave_sync();
                    continue;
                }
                bool take = status != UQK_STATUS_LINE_SEARCH;
                if (lagged) {
                    // a lagged direction is not halved: it is kept when the
                    // full step lowers ||grad L|| (the FP64 accept test), else
                    // lambda stays and the next iteration factors its own
                    // Hessian and runs the reference Newton step
                    take = nt < ng;
                    if (take) {
                        ++w_count[6];
                        // contraction clearly worse than a (damped) Newton
                        // step's: factor afresh at the next Newton step
                        if (!(nt / ng <= 1.2 * (1.0 - c.alpha) + 1e-3)) refactor = true;
                    } else {
#pragma unroll
                        for (int s = 0; s < S; ++s) Lk[s] = Lk0[s];
                        rk = rk0;
                        refactor = true;
                    }
                }
                if (take) {
                    double* t = lam;
                    lam = lamnew;
                    lamnew = t;
                    ub_lam = true;
                    ng = nt;
                    g = gt;
                    if (status < 0 && !lagged && !isfinite(nt)) status = UQK_STATUS_NONFINITE;
                    if (status < 0 && nt < c.eps) status = UQK_STATUS_CONVERGED;
                }
            } else {
                if (where == ALT) {
                    // learned start: Newton starts from the candidate with the
                    // smaller ||grad L|| (a NaN norm fails the comparison and
                    // never wins)
                    if (nt < ng) {
                        double* t = lam;
                        lam = lamnew;
                        lamnew = t;
                        g = gt;
                        ng = nt;
                        ++w_count[4];
                        ub_lam = true;
                    } else {
                        ub_lam = false;
                        g = g0;
#pragma unroll
                        for (int s = 0; s < S; ++s) Lk[s] = Lk0[s];
                        rk = rk0;
                    }
                } else {
                    if (where == START) {
                        g = gt;
                        ng = nt;
                        ub_lam = true;
                    }
                    if (a.lam_alt && (c.safe || !(ng < c.eps))) {
                        if (on) lamnew[dj] = la_c;
                        g0 = g;
#pragma unroll
                        for (int s = 0; s < S; ++s) Lk0[s] = Lk[s];
                        rk0 = rk;
                        wave_sync();
                        where = ALT;
                        at = lamnew;
                        continue;
                    }
                }
                if (!c.safe && ng < c.eps) status = UQK_STATUS_CONVERGED;
            }
            if (status < 0 && iters >= c.max_iter) status = UQK_STATUS_MAX_ITERATIONS;
            if (status < 0) {
                // the next Newton direction
                ++iters;
                // a lagged step (mixed precision, kept inverse P): d = P g --
                // across time steps with one step of iterative refinement
                // against the FP64 Hessian at lambda, d += P (g - H d)
                if constexpr (wave_reuses<PREC>) lagged = reuse && !refactor;
                if (lagged) {
                    if constexpr (PREC == 4) d = apply_inverse(T_call, g);
                    if constexpr (PREC == 2) {
                        const double d1 = pmatvec(g);
                        const double hv = hessvec(d1);
                        d = d1 + pmatvec(g - hv);
                    }
#pragma unroll
                    for (int s = 0; s < S; ++s) Lk0[s] = Lk[s];
                    rk0 = rk;
                } else {
                    bool spd;
                    if constexpr (PREC == 2) {
                        // phase: factor
                        spd = sweep_step<KIND, M, Q>(c, Lk[0], Lk[S > 1 ? 1 : 0], Lk[S > 2 ? 2 : 0],
                                                     Lk[S > 3 ? 3 : 0], rk, g, (lds_double*)smem, (lds_double*)wb,
                                                     reuse ? a.pinv + cell * (long)W::KEPT : nullptr);
                        // phase end: factor
                        d = on ? yb[de] : 0.0;
                        wave_sync();
                        if (spd && reuse) factored = true;
                        // a cell that factors applies no kept inverse after
                        // it (said here for the registers' sake)
#pragma unroll
                        for (int r = 0; r < KT; ++r)
#pragma unroll
                            for (int t = 0; t < KQ; ++t) kept[r][t] = 0.f;
                    } else {
                        renew();
                        // phase: hessian
                        wave_system<KIND, M, Q, PREC == 0>(c, Lk, rk, g, smem, bh, lane, p16, q4);
                        // phase end: hessian
                        if constexpr (PREC == 4) {
                            load_system(T_call);
                            // phase: factor
                            spd = tile_sweep<NT>(T_call, N, p16, q4);
                            // phase end: factor
                            if (spd) d = apply_inverse(T_call, g);
                            refactor = false;
                        } else {
                            f64x4 T[TILES];
                            load_system(T);
                            // phase: factor
                            spd = tile_ldl<NT>(T, N, p16, q4);
                            // phase end: factor
                            // phase: backsub
                            if (spd) d = to_duals(tile_back<NT>(T, N, p16, q4));
                            // phase end: backsub
                        }
                    }
                    if (!spd) {
                        status = UQK_STATUS_NOT_SPD;
                    } else {
                        ++w_count[5];
                        if (c.max_iter == 1) {  // one-shot IPM (closure.cpp:151-154)
                            if (on) lam[dj] -= c.alpha * d;
                            ub_lam = false;
                            wave_sync();
                            status = UQK_STATUS_CONVERGED;
                        }
                    }
                }
            }
            if (kEarly && resolved < 2) {
                next = queue.take();
                prefetch(next);
                resolved = 2;
            }
            if (status < 0) {
                step = 1.0;
                halvings = 0;
                if (on) lamnew[dj] = lam[dj] - step * c.alpha * d;
                wave_sync();
                where = TRIAL;
                at = lamnew;
                continue;
            }
            // the outputs come from U at the returned lambda: evaluated again
            // where the last gradient was another point's (a rejected step, a
            // failed cell, or the check's gradient alone)
            if (!a.uq_out || ub_lam) break;
            where = END;
            at = lam;
        }
        // phase: outputs
        if constexpr (!kEarly) {
            next = queue.take();
            prefetch(next);
        }
        arrive();
        // the cell's slot for the next launch: a usable inverse (1) -- the
        // one just stored, or the kept one while it is fresh -- or none (0)
        if (PREC == 2 && reuse && lane == 0) a.pinv_ok[cell] = factored || !refactor ? 1 : 0;
        if (on) lg[dj] = lam[dj];
        if (a.uq_out) {
            // the step's next two sweeps, from the last gradient at the
            // returned lambda: uQ = U(lambda phi) (momentsolver.cpp:100) and
            // u = <uQ phiW> (:120-124)
            double* uqg = a.uq_out + cell * (long)Q * S;
            for (int t = lane; t < Q * S; t += 64) {
                const int k = t / S, s = t - k * S;
                uqg[t] = Ub[s * QP + k];
            }
            if (on) a.u_out[cell * SM + dj] = uproj;
            if (a.dt_min) {  // momentsolver.cpp:127-133 for this cell
                double m = 1e10;
                if (lane < Q) {
                    double uk[S];
#pragma unroll
                    for (int s = 0; s < S; ++s) uk[s] = Ub[s * QP + lane];
                    m = point_dt<S>(a.dtp, uk, dx_c);
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
        // status, iters and ngrad are wave-uniform: these sums stay scalar
        w_count[1] += status != UQK_STATUS_CONVERGED ? 1ull : 0ull;
        w_count[2] += (unsigned long long)iters;
        w_count[3] += (unsigned long long)ngrad;
        wave_sync();
        // phase end: outputs
    }
    add_counts(w_count, w_dt, smem, a.counter, a.dt_min);
}

// ---------------------------------------------------------------------------
// dispatch over the compiled shapes
// ---------------------------------------------------------------------------
template <int KIND, int M, int Q, int PREC>
static size_t wave_lds(int waves) {
    using W = WaveShape<KIND, M, Q>;
    return sizeof(double) * (W::ADDR + wave_tiles<PREC, W::NT> * 64 + (size_t)waves * W::WAVE_DOUBLES);
}

template <int KIND, int M, int Q, int PREC>
static int wave_max_waves(int max_lds) {
    int waves = 4;
    while (waves > 1 && wave_lds<KIND, M, Q, PREC>(waves) > (size_t)max_lds) --waves;
    return waves;
}

template <int KIND, int M, int Q, int PREC>
static int wave_occupancy(int waves) {
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, newton_wave_kernel<KIND, M, Q, PREC>, 64 * waves,
                                                     wave_lds<KIND, M, Q, PREC>(waves)) != hipSuccess ||
        occ <= 0)
        occ = 1;
    return occ;
}

template <int KIND, int M, int Q, int PREC>
static void wave_go(const NewtonArgs& a, int max_lds, int num_cu, hipStream_t st, hipError_t* err,
                    const LaunchShape& shape) {
    const int wmax = wave_max_waves<KIND, M, Q, PREC>(max_lds);
    int waves = shape.waves > 0 ? (shape.waves < wmax ? shape.waves : wmax) : wmax;
    const int threads = 64 * waves;
    const size_t shmem = wave_lds<KIND, M, Q, PREC>(waves);
    const int occ = wave_occupancy<KIND, M, Q, PREC>(waves);
    const int per_cu = shape.blocks_per_cu > 0 && shape.blocks_per_cu < occ ? shape.blocks_per_cu : occ;
    long want = (a.ncell + waves - 1) / waves;
    int blocks = (int)(want < (long)per_cu * num_cu ? want : (long)per_cu * num_cu);
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL((newton_wave_kernel<KIND, M, Q, PREC>), dim3(blocks), dim3(threads), shmem, st, a);
    *err = hipGetLastError();
}

template <int KIND, int M, int Q>
static bool wave_fits(int kind, int m, int q, int max_lds) {
    if (kind != KIND || m != M || q != Q) return false;
    return wave_lds<KIND, M, Q, 4>(1) <= (size_t)max_lds;  // (PREC 4 holds the most tiles)
}

}  // namespace uqk
