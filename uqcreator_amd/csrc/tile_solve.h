// tile_solve.h -- factorisation, solve and inversion of a symmetric positive
// definite system by one wavefront, entirely in registers.
//
// The matrix lies in 16 x 16 tiles in the accumulator layout of
// v_mfma_f64_16x16x4f64: element e (0..3) of lane 16 q + p of tile (tc, tr)
// is H(r = 16 tr + p, c = 16 tc + 4 e + q).  In that layout the four columns
// c = 4 b .. 4 b + 3 of a tile row are ONE register (lane group q holds column
// 4 b + q of row p), and this register is, as it stands, the A operand (rows
// p, k = q) and the B operand (k = q, columns p) of a rank-4 update.  So four
// pivots are eliminated per step without moving the panel:
//   B   = L D L^T, the 4 x 4 pivot block, factored by every lane from
//         v_readlane'd scalars (four reciprocals in sequence, of which V
//         waits for three);
//   V   = P L^-T, one v_mfma_f64_4x4x4_4b per 16 rows of the panel P;
//   H  -= V D^-1 V^T on the tiles that are left, one v_mfma_f64_16x16x4 each.
// There is no LDS round trip and no lane mask per entry.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "uqk_device.h"

namespace uqk {

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double lane_get(double v, int lane) {
    const long long x = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)x, lane);
    const int hi = __builtin_amdgcn_readlane((int)(x >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const long long x = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(x >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// sum over each row of 16 lanes, in every lane (DPP row rotations)
__device__ __forceinline__ double row_sum(double v) {
    v += dpp_f64<0x128>(v);  // row_ror:8
    v += dpp_f64<0x124>(v);
    v += dpp_f64<0x122>(v);
    v += dpp_f64<0x121>(v);
    return v;
}

// sum over the four lanes that share p, in every lane (gfx950 row swaps)
__device__ __forceinline__ double group_sum(double v) {
    const long long x = __double_as_longlong(v);
    const auto l16 = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)x, false, false);
    const auto h16 = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(x >> 32), false, false);
    const double s = __longlong_as_double(((long long)h16[0] << 32) | (unsigned)l16[0]) +
                     __longlong_as_double(((long long)h16[1] << 32) | (unsigned)l16[1]);
    const long long y = __double_as_longlong(s);
    const auto l32 = __builtin_amdgcn_permlane32_swap((unsigned)y, (unsigned)y, false, false);
    const auto h32 = __builtin_amdgcn_permlane32_swap((unsigned)(y >> 32), (unsigned)(y >> 32), false, false);
    return __longlong_as_double(((long long)h32[0] << 32) | (unsigned)l32[0]) +
           __longlong_as_double(((long long)h32[1] << 32) | (unsigned)l32[1]);
}

__device__ __forceinline__ void swap_halves(double& a, double& b) {  // a's lanes 32..63 with b's lanes 0..31
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    a = __longlong_as_double(((long long)hi[0] << 32) | (unsigned)lo[0]);
    b = __longlong_as_double(((long long)hi[1] << 32) | (unsigned)lo[1]);
}
__device__ __forceinline__ void swap_rows(double& a, double& b) {  // a's odd rows of 16 lanes with b's even ones
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    a = __longlong_as_double(((long long)hi[0] << 32) | (unsigned)lo[0]);
    b = __longlong_as_double(((long long)hi[1] << 32) | (unsigned)lo[1]);
}
// register t of lane group s <-> register s of lane group t
__device__ __forceinline__ void group_transpose(double (&d)[4]) {
    swap_halves(d[0], d[2]);
    swap_halves(d[1], d[3]);
    swap_rows(d[0], d[1]);
    swap_rows(d[2], d[3]);
}

// basis pair (j <= i) of number e = i (i + 1) / 2 + j, from its root (e < 2^14)
__device__ __forceinline__ void basis_pair(int e, int& j, int& i) {
    i = (int)((__builtin_amdgcn_sqrtf(8.f * (float)e + 1.f) - 1.f) * 0.5f);
    const int below = (int)__umul24(i, i + 1) >> 1;  // (24-bit products: the 32-bit one takes four times as long)
    const int low = below > e ? 1 : 0, high = below + i + 1 <= e ? 1 : 0;
    j = e - (below - (low ? i : 0) + (high ? i + 1 : 0));
    i += high - low;
}

// Stands where paths join that matrix instructions precede on some of them.
// What reads their results has to come 9 (4 x 4 x 4) or 18 (16 x 16 x 4) issue
// slots later at most; the compiler counts these slots along one of the paths
// to a join only, and where a shorter one exists the read can come too early
// (seen as the old low half of a result).
template <int SLOTS>
__device__ __forceinline__ void settle() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop %0" : : "n"(SLOTS < 16 ? SLOTS - 1 : 15));
    if constexpr (SLOTS > 16) asm volatile("s_nop %0" : : "n"(SLOTS - 17));
    __builtin_amdgcn_sched_barrier(0);
}

// mma(load(0)), mma(load(1)), .. for `steps` steps, U of them in flight: the
// next U are loaded while these are multiplied (what an LDS round trip costs
// a wavefront with no other beside it, or few).  Steps are loaded up to U past
// the last, so the operands' rows need that much readable LDS behind them.
// (Written out, because loops over matrix instructions are not unrolled with a
// remainder.)
template <int U, class Load, class Mma>
__device__ __forceinline__ void in_steps(int steps, Load load, Mma mma) {
    decltype(load(0)) x[U], y[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = load(u);
    int s = 0;
    for (; s + 2 * U < steps; s += 2 * U) {
#pragma unroll
        for (int u = 0; u < U; ++u) y[u] = load(s + U + u);
#pragma unroll
        for (int u = 0; u < U; ++u) mma(x[u]);
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = load(s + 2 * U + u);
#pragma unroll
        for (int u = 0; u < U; ++u) mma(y[u]);
    }
    if (s + U < steps) {
#pragma unroll
        for (int u = 0; u < U; ++u) y[u] = load(s + U + u);
#pragma unroll
        for (int u = 0; u < U; ++u) mma(x[u]);
        s += U;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s + u < steps) mma(y[u]);
    } else {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s + u < steps) mma(x[u]);
    }
    settle<9>();
}
// Operands of a matrix step, and of two steps: eight points, of which lane
// group q holds 2 q and 2 q + 1 (one ds_read_b128 each; 16 rows of 4 mod 8
// doubles at these four columns fall on all 64 banks once: 8.8 cycles per
// double and lane with four wavefronts, where ds_read_b64 of rows 4 mod 8 at
// columns q takes 64 and of odd rows 16).
typedef double f64x2 __attribute__((ext_vector_type(2)));
template <int N, class T = double>
struct Operands {
    T a, b[N];
};
__device__ __forceinline__ f64x2 two(const double* x) { return *reinterpret_cast<const f64x2*>(x); }

// f(integral_constant<0>) .. f(integral_constant<N - 1>)
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        static_for<N, I + 1>(f);
    }
}

// tile (tc, tr), tc <= tr, of the lower triangle
__host__ __device__ constexpr int tile_lower(int tc, int tr) { return tr * (tr + 1) / 2 + tc; }

// The 4 x 4 pivot block B = L D L^T at row/column j0 (0, 4, 8, 12) of a
// diagonal tile whose panel register is pv, formed by every lane from
// v_readlane'd scalars: lane 16 q + p gets li = L^-1(p % 4, q), lt = L^-1(q, p
// % 4) and di = 1/D(q).  Of the four pivots only `have` are real, the others
// read as identity.  False if a pivot is not positive.
// The factors and not B^-1, because the update with V = P L^-T, H -= V D^-1
// V^T, stands as much ill-conditioning as the Cholesky factorisation does;
// with H -= P B^-1 P^T the Newton iteration met pivots that rounding had made
// negative in 23 of 40 Euler closures that Cholesky solves (n = 40, a start of
// a far too small density).  No product of two pivots either: it underflows
// where the density does.  Both cost nothing: 65,536 cells of n = 40, 40 time
// steps in FP64, 20.1 ms against 20.5 with the inverse from two 2 x 2 blocks.
__device__ __forceinline__ bool pivot_factors(double pv, int j0, int have, int p, int q, double& li, double& lt,
                                              double& di) {
    double b00 = lane_get(pv, j0), b10 = lane_get(pv, j0 + 1), b20 = lane_get(pv, j0 + 2), b30 = lane_get(pv, j0 + 3);
    double b11 = lane_get(pv, 16 + j0 + 1), b21 = lane_get(pv, 16 + j0 + 2), b31 = lane_get(pv, 16 + j0 + 3);
    double b22 = lane_get(pv, 32 + j0 + 2), b32 = lane_get(pv, 32 + j0 + 3), b33 = lane_get(pv, 48 + j0 + 3);
    if (have < 4) {
        b33 = 1.0, b30 = b31 = b32 = 0.0;
        if (have < 3) b22 = 1.0, b20 = b21 = 0.0;
        if (have < 2) b11 = 1.0, b10 = 0.0;
    }
    const double r0 = recip_f64(b00), l10 = b10 * r0, l20 = b20 * r0, l30 = b30 * r0;
    const double d1 = fma(-l10, b10, b11), c21 = fma(-l20, b10, b21), c31 = fma(-l30, b10, b31);
    const double r1 = recip_f64(d1), l21 = c21 * r1, l31 = c31 * r1;
    const double d2 = fma(-l21, c21, fma(-l20, b20, b22)), c32 = fma(-l31, c21, fma(-l30, b20, b32));
    const double r2 = recip_f64(d2), l32 = c32 * r2;
    const double d3 = fma(-l32, c32, fma(-l31, c31, fma(-l30, b30, b33)));
    const double r3 = recip_f64(d3);
    // L^-1: i10 = -l10, i21 = -l21, i32 = -l32
    const double i20 = fma(l21, l10, -l20), i31 = fma(l32, l21, -l31);
    const double i30 = fma(-l32, i20, fma(l31, l10, -l30));
    const bool p1 = p & 1, p2 = p & 2, q1 = q & 1, q2 = q & 2;
    const double c0 = p2 ? (p1 ? i30 : i20) : (p1 ? -l10 : 1.0);
    const double c1 = p2 ? (p1 ? i31 : -l21) : (p1 ? 1.0 : 0.0);
    const double c2 = p2 ? (p1 ? -l32 : 1.0) : 0.0, c3 = p1 && p2 ? 1.0 : 0.0;
    li = q2 ? (q1 ? c3 : c2) : (q1 ? c1 : c0);
    lt = __builtin_amdgcn_mfma_f64_4x4x4f64(li, (p & 3) == q ? 1.0 : 0.0, 0.0, 0, 0, 0);  // (transposed)
    di = q2 ? (q1 ? r3 : r2) : (q1 ? r1 : r0);
    return b00 > 0.0 && d1 > 0.0 && d2 > 0.0 && d3 > 0.0;
}

// In place on the lower tiles of [H; g^T] (n pivots; row n holds the right
// hand side): column block b becomes V D^-1, that of the unit lower factor of
// H = L D L^T, and the block's own rows its L^-1, transposed.  The first NT
// tile rows hold n + 1 rows; there is no branch between the matrix
// instructions of a step, whose tiles past the last pivot are updated for
// nothing where n is not a constant (settle).
template <int NT, int TILES>
__device__ __forceinline__ bool tile_ldl(f64x4 (&T)[TILES], int n, int p, int q) {
    bool ok = true;
#pragma unroll
    for (int b = 0; b < 4 * NT; ++b) {
        if (4 * b >= n) break;
        const int jb = b >> 2, e = b & 3, j0 = 4 * e, have = n - 4 * b;
        double li, lt, di;
        ok &= pivot_factors(T[tile_lower(jb, jb)][e], j0, have, p, q, li, lt, di);
        double V[NT], W[NT];
#pragma unroll
        for (int r = jb; r < NT; ++r) {
            double P = T[tile_lower(jb, r)][e];
            if (r == jb && !(p >= j0 + (have < 4 ? have : 4))) P = 0.0;  // finished rows
            if (have < 4 && q >= have) P = 0.0;                          // columns that are no pivots
            V[r] = __builtin_amdgcn_mfma_f64_4x4x4f64(li, P, 0.0, 0, 0, 0);
            W[r] = V[r] * di;
            T[tile_lower(jb, r)][e] = r == jb && (p >> 2) == e && (p & 3) < have ? lt : W[r];
        }
        if (!__builtin_constant_p(n) || 4 * b + 4 < n) {
#pragma unroll
            for (int r = jb; r < NT; ++r)
#pragma unroll
                for (int c = jb; c <= r; ++c)
                    if (!__builtin_constant_p(n) || 16 * c < n)
                        T[tile_lower(c, r)] =
                            __builtin_amdgcn_mfma_f64_16x16x4f64(V[c], -W[r], T[tile_lower(c, r)], 0, 0, 0);
        }
    }
    if (!__builtin_constant_p(n)) settle<18>();
    return ok;
}

// The solution from the factor that tile_ldl left, four unknowns per step:
// y_k = (V D^-1)(n, k) - sum_{r > 4b+3} (V D^-1)(r, k) x_r, the sum over the
// rows of a lane group by DPP, and x = L^-T y of the block over the lane
// groups.  X[r] of lane 16 q + p is x_{16 r + p} (-1 at n, zero past it).
template <int NT, int TILES>
__device__ __forceinline__ void tile_back_rows(const f64x4 (&T)[TILES], int n, int p, int q, double (&X)[NT]) {
#pragma unroll
    for (int r = 0; r < NT; ++r) X[r] = 16 * r + p == n ? -1.0 : 0.0;
#pragma unroll
    for (int b = 4 * NT - 1; b >= 0; --b) {
        if (4 * b >= n) continue;
        const int jb = b >> 2, e = b & 3, have = n - 4 * b;
        double s = 0.0;
#pragma unroll
        for (int r = jb; r < NT; ++r)
            s = fma(-T[tile_lower(jb, r)][e], X[r], s);
        const double x = group_sum(T[tile_lower(jb, jb)][e] * row_sum(s));
        if ((p >> 2) == e && (p & 3) < have) X[jb] = x;
    }
}

// The same for n < 64: lane l gets x_l (zero past n).
template <int NT, int TILES>
__device__ __forceinline__ double tile_back(const f64x4 (&T)[TILES], int n, int p, int q) {
    double X[NT];
    tile_back_rows<NT>(T, n, p, q, X);
    double d = X[0];
#pragma unroll
    for (int r = 1; r < NT; ++r) d = q == r ? X[r] : d;
    return 16 * q + p < n ? d : 0.0;
}

// In place on all NT x NT tiles (tile (tc, tr) at tr * NT + tc): the sweep
// of every pivot block, which leaves -H^-1 in the rows and columns below n
// and H^-1 g in column n (where row and column n held the right-hand side).
// The pivot columns, set to zero beforehand, get P B^-1, and -B^-1 in the block
// itself, from the same products: -L^-T stands in the place of V's pivot rows.
template <int NT>
__device__ __forceinline__ bool tile_sweep(f64x4 (&T)[NT * NT], int n, int p, int q) {
    bool ok = true;
#pragma unroll
    for (int b = 0; b < 4 * NT; ++b) {
        if (4 * b >= n) break;
        const int jb = b >> 2, e = b & 3, have = n - 4 * b;
        double li, lt, di;
        ok &= pivot_factors(T[jb * NT + jb][e], 4 * e, have, p, q, li, lt, di);
        const bool in = (p >> 2) == e && (p & 3) < have;  // this lane's row of tile row jb is a pivot
        double V[NT], U[NT];
#pragma unroll
        for (int r = 0; r < NT; ++r) {
            double P = T[r * NT + jb][e];
            if (r == jb && in) P = 0.0;
            if (have < 4 && q >= have) P = 0.0;
            V[r] = __builtin_amdgcn_mfma_f64_4x4x4f64(li, P, 0.0, 0, 0, 0);
            if (r == jb && in) V[r] = -lt;
            U[r] = V[r] * di;
            if (!(have < 4 && q >= have)) T[r * NT + jb][e] = 0.0;
        }
        if (in) {
#pragma unroll
            for (int c = 0; c < NT; ++c) T[jb * NT + c] = f64x4{0.0, 0.0, 0.0, 0.0};
        }
#pragma unroll
        for (int r = 0; r < NT; ++r)
#pragma unroll
            for (int c = 0; c < NT; ++c)
                T[r * NT + c] = __builtin_amdgcn_mfma_f64_16x16x4f64(V[c], -U[r], T[r * NT + c], 0, 0, 0);
    }
    return ok;
}

// The same sweep on the lower tiles alone (two thirds of the registers and
// of the matrix steps at NT = 3): the panel's rows above the pivots are the
// transposed pivot rows, turned over through LDS (scr, 64 (NT - 1) doubles).
// -H^-1 in the lower triangle, and H^-1 g in row n where row n held g.
template <int NT, int TILES, class D>
__device__ __forceinline__ bool tile_sweep_lower(f64x4 (&T)[TILES], int n, int p, int q, D* scr) {
    bool ok = true;
#pragma unroll
    for (int b = 0; b < 4 * NT; ++b) {
        if (4 * b >= n) break;
        const int jb = b >> 2, e = b & 3, have = n - 4 * b;
        double li, lt, di;
        const bool at = (p >> 2) == e;
        if (jb > 0) {
            wave_sync();
            if (at) {
#pragma unroll
                for (int r = 0; r < jb; ++r)
#pragma unroll
                    for (int h = 0; h < 4; ++h) scr[64 * r + 16 * (p & 3) + 4 * h + q] = T[tile_lower(r, jb)][h];
            }
            wave_sync();
        }
        ok &= pivot_factors(T[tile_lower(jb, jb)][e], 4 * e, have, p, q, li, lt, di);
        const bool in = at && (p & 3) < have;  // this lane's row of tile row jb is a pivot
        double V[NT];
#pragma unroll
        for (int r = 0; r < NT; ++r) {
            double P = r < jb ? scr[64 * r + 16 * q + p] : T[tile_lower(jb, r < jb ? jb : r)][e];
            if (r == jb && in) P = 0.0;
            if (have < 4 && q >= have) P = 0.0;
            V[r] = __builtin_amdgcn_mfma_f64_4x4x4f64(li, P, 0.0, 0, 0, 0);
            if (r == jb && in) V[r] = -lt;
        }
        if (in) {
#pragma unroll
            for (int c = 0; c <= jb; ++c) T[tile_lower(c, jb)] = f64x4{0.0, 0.0, 0.0, 0.0};
        }
#pragma unroll
        for (int r = 0; r < NT; ++r) {
            const double U = V[r] * di;
            if (jb <= r && !(have < 4 && q >= have)) T[tile_lower(jb <= r ? jb : r, r)][e] = 0.0;
#pragma unroll
            for (int c = 0; c <= r; ++c)
                T[tile_lower(c, r)] = __builtin_amdgcn_mfma_f64_16x16x4f64(V[c], -U, T[tile_lower(c, r)], 0, 0, 0);
        }
    }
    if (!__builtin_constant_p(n)) settle<18>();
    return ok;
}

}  // namespace uqk
