// tile_solve.h -- factorisation, solve and inversion of a symmetric positive
// definite system of n < 64 unknowns by one wavefront, entirely in registers.
//
// The matrix lies in 16 x 16 tiles in the accumulator layout of
// v_mfma_f64_16x16x4f64: element e (0..3) of lane 16 q + p of tile (tc, tr)
// is H(r = 16 tr + p, c = 16 tc + 4 e + q).  In that layout the four columns
// c = 4 b .. 4 b + 3 of a tile row are ONE register (lane group q holds column
// 4 b + q of row p), and this register is, as it stands, the A operand (rows
// p, k = q) and the B operand (k = q, columns p) of a rank-4 update.  So four
// pivots are eliminated per step without moving the panel:
//   B   = the 4 x 4 pivot block, inverted by every lane from v_readlane'd
//         scalars (two 2 x 2 blocks, so two reciprocals are in sequence, not
//         four);
//   W   = P B^-1, one v_mfma_f64_4x4x4_4b per 16 rows of the panel P;
//   H  -= P W^T on the tiles that are left, one v_mfma_f64_16x16x4 each.
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

// B^-1 of the 4 x 4 pivot block at row/column j0 (0, 4, 8, 12) of a diagonal
// tile whose panel register is pv; lane 16 q + p gets B^-1(p % 4, q).  Of
// the four pivots only `have` are real, the others read as identity.  False
// if a leading minor is not positive.
__device__ __forceinline__ bool pivot_inverse(double pv, int j0, int have, int p, int q, double& bv) {
    double b00 = lane_get(pv, j0), b10 = lane_get(pv, j0 + 1), b20 = lane_get(pv, j0 + 2), b30 = lane_get(pv, j0 + 3);
    double b11 = lane_get(pv, 16 + j0 + 1), b21 = lane_get(pv, 16 + j0 + 2), b31 = lane_get(pv, 16 + j0 + 3);
    double b22 = lane_get(pv, 32 + j0 + 2), b32 = lane_get(pv, 32 + j0 + 3), b33 = lane_get(pv, 48 + j0 + 3);
    if (have < 4) {
        b33 = 1.0, b30 = b31 = b32 = 0.0;
        if (have < 3) b22 = 1.0, b20 = b21 = 0.0;
        if (have < 2) b11 = 1.0, b10 = 0.0;
    }
    // E = [b00 b10; b10 b11] = L D L^T; 1/d1 = b00 / det, so that both
    // reciprocals start at once
    const double det = fma(b00, b11, -b10 * b10);
    const double r0 = recip_f64(b00), e11 = b00 * recip_f64(det), l = b10 * r0;
    const double e01 = -l * e11, e00 = fma(-l, e01, r0);
    // X = E^-1 F, F = [b20 b30; b21 b31]; S = G - F^T X
    const double x00 = fma(e00, b20, e01 * b21), x10 = fma(e01, b20, e11 * b21);
    const double x01 = fma(e00, b30, e01 * b31), x11 = fma(e01, b30, e11 * b31);
    const double s00 = fma(-b20, x00, fma(-b21, x10, b22));
    const double s10 = fma(-b20, x01, fma(-b21, x11, b32));
    const double s11 = fma(-b30, x01, fma(-b31, x11, b33));
    const double dets = fma(s00, s11, -s10 * s10);
    const double t0 = recip_f64(s00), i33 = s00 * recip_f64(dets), m = s10 * t0;
    const double i23 = -m * i33, i22 = fma(-m, i23, t0);
    // Y = X S^-1
    const double y00 = fma(x00, i22, x01 * i23), y01 = fma(x00, i23, x01 * i33);
    const double y10 = fma(x10, i22, x11 * i23), y11 = fma(x10, i23, x11 * i33);
    const double i00 = fma(y00, x00, fma(y01, x01, e00)), i01 = fma(y00, x10, fma(y01, x11, e01));
    const double i11 = fma(y10, x10, fma(y11, x11, e11));
    const int pm = p & 3;
    // row pm of the symmetric inverse: columns q
    const bool p1 = pm & 1, p2 = pm & 2, q1 = q & 1, q2 = q & 2;
    const double c0 = q1 ? (p1 ? i11 : i01) : (p1 ? i01 : i00);      // p, q < 2
    const double c2 = q1 ? (p1 ? i33 : i23) : (p1 ? i23 : i22);      // p, q >= 2
    // -Y(a, b): row a < 2 and column 2 + b
    const bool a1 = p2 ? q1 : p1, d1 = p2 ? p1 : q1;
    const double c1 = -(d1 ? (a1 ? y11 : y01) : (a1 ? y10 : y00));
    bv = p2 == q2 ? (p2 ? c2 : c0) : c1;
    return b00 > 0.0 && det > 0.0 && s00 > 0.0 && dets > 0.0;
}

// In place on the lower tiles of [H; g^T] (n pivots; row n holds the right
// hand side): column block b becomes W = V^T, the block-unit upper factor of
// H = V^T B V (B the 4 x 4 pivot blocks).  The first NT tile rows hold n + 1
// rows; there is no branch between the matrix instructions of a step, whose
// tiles past the last pivot are updated for nothing where n is not a constant
// (settle).
template <int NT, int TILES>
__device__ __forceinline__ bool tile_ldl(f64x4 (&T)[TILES], int n, int p, int q) {
    bool ok = true;
#pragma unroll
    for (int b = 0; b < 4 * NT; ++b) {
        if (4 * b >= n) break;
        const int jb = b >> 2, e = b & 3, j0 = 4 * e, have = n - 4 * b;
        double bv;
        ok &= pivot_inverse(T[tile_lower(jb, jb)][e], j0, have, p, q, bv);
        double P[NT], W[NT];
#pragma unroll
        for (int r = jb; r < NT; ++r) {
            P[r] = T[tile_lower(jb, r)][e];
            if (r == jb && !(p >= j0 + (have < 4 ? have : 4))) P[r] = 0.0;  // finished rows
            if (have < 4 && q >= have) P[r] = 0.0;       // columns that are no pivots
            W[r] = __builtin_amdgcn_mfma_f64_4x4x4f64(bv, P[r], 0.0, 0, 0, 0);
            T[tile_lower(jb, r)][e] = W[r];
        }
        if (!__builtin_constant_p(n) || 4 * b + 4 < n) {
#pragma unroll
            for (int r = jb; r < NT; ++r)
#pragma unroll
                for (int c = jb; c <= r; ++c)
                    if (!__builtin_constant_p(n) || 16 * c < n)
                        T[tile_lower(c, r)] =
                            __builtin_amdgcn_mfma_f64_16x16x4f64(P[c], -W[r], T[tile_lower(c, r)], 0, 0, 0);
        }
    }
    if (!__builtin_constant_p(n)) settle<18>();
    return ok;
}

// The solution from the factor that tile_ldl left: x_{4b+k} = W(n, k) -
// sum_{r > 4b+3} W(r, k) x_r, four unknowns per step, the sum over the rows
// of a lane group by DPP.  X[r] of lane 16 q + p is x_{16 r + p} (-1 at n,
// zero past it).
template <int NT, int TILES>
__device__ __forceinline__ void tile_back_rows(const f64x4 (&T)[TILES], int n, int p, int q, double (&X)[NT]) {
#pragma unroll
    for (int r = 0; r < NT; ++r) X[r] = 16 * r + p == n ? -1.0 : 0.0;
    const bool p1 = p & 1, p2 = p & 2;
#pragma unroll
    for (int b = 4 * NT - 1; b >= 0; --b) {
        if (4 * b >= n) continue;
        const int jb = b >> 2, e = b & 3, have = n - 4 * b;
        double s = 0.0;
#pragma unroll
        for (int r = jb; r < NT; ++r)
            s = fma(-T[tile_lower(jb, r)][e], X[r], s);
        s = row_sum(s);
        const double x0 = lane_get(s, 0), x1 = lane_get(s, 16), x2 = lane_get(s, 32), x3 = lane_get(s, 48);
        const double v = p2 ? (p1 ? x3 : x2) : (p1 ? x1 : x0);
        if ((p >> 2) == e && (p & 3) < have) X[jb] = v;
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
template <int NT>
__device__ __forceinline__ bool tile_sweep(f64x4 (&T)[NT * NT], int n, int p, int q) {
    bool ok = true;
#pragma unroll
    for (int b = 0; b < 4 * NT; ++b) {
        if (4 * b >= n) break;
        const int jb = b >> 2, e = b & 3, have = n - 4 * b;
        double bv;
        ok &= pivot_inverse(T[jb * NT + jb][e], 4 * e, have, p, q, bv);
        const bool in = (p >> 2) == e && (p & 3) < have;  // this lane's row of tile row jb is a pivot
        double P[NT], W[NT], R[NT];
#pragma unroll
        for (int r = 0; r < NT; ++r) {
            P[r] = T[r * NT + jb][e];
            if (r == jb && in) P[r] = 0.0;
            if (have < 4 && q >= have) P[r] = 0.0;
            W[r] = __builtin_amdgcn_mfma_f64_4x4x4f64(bv, P[r], 0.0, 0, 0, 0);
            // pivot rows: H(c, pivot) <- W(c, .) = sum_k P(c, k) B^-1(k, .)
            R[r] = r == jb && in ? bv : -W[r];
        }
        if (in) {
#pragma unroll
            for (int c = 0; c < NT; ++c) T[jb * NT + c] = f64x4{0.0, 0.0, 0.0, 0.0};
        }
#pragma unroll
        for (int r = 0; r < NT; ++r)
#pragma unroll
            for (int c = 0; c < NT; ++c) {
                const double old = T[r * NT + c][e];
                T[r * NT + c] = __builtin_amdgcn_mfma_f64_16x16x4f64(P[c], R[r], T[r * NT + c], 0, 0, 0);
                if (c == jb) {
                    // the pivot columns: W, and -B^-1 in the block itself
                    const double w = r == jb && in ? -bv : W[r];
                    T[r * NT + c][e] = have < 4 && q >= have ? old : w;
                }
            }
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
        double bv;
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
        ok &= pivot_inverse(T[tile_lower(jb, jb)][e], 4 * e, have, p, q, bv);
        const bool in = at && (p & 3) < have;  // this lane's row of tile row jb is a pivot
        double P[NT], W[NT];
#pragma unroll
        for (int r = 0; r < NT; ++r) {
            P[r] = r < jb ? scr[64 * r + 16 * q + p] : T[tile_lower(jb, r < jb ? jb : r)][e];
            if (r == jb && in) P[r] = 0.0;
            if (have < 4 && q >= have) P[r] = 0.0;
        }
        if (in) {
#pragma unroll
            for (int c = 0; c <= jb; ++c) T[tile_lower(c, jb)] = f64x4{0.0, 0.0, 0.0, 0.0};
        }
#pragma unroll
        for (int r = 0; r < NT; ++r) {
            W[r] = __builtin_amdgcn_mfma_f64_4x4x4f64(bv, P[r], 0.0, 0, 0, 0);
            const double R = r == jb && in ? bv : -W[r];
#pragma unroll
            for (int c = 0; c <= r; ++c) {
                const double old = T[tile_lower(c, r)][e];
                T[tile_lower(c, r)] = __builtin_amdgcn_mfma_f64_16x16x4f64(P[c], R, T[tile_lower(c, r)], 0, 0, 0);
                if (c == jb) {
                    const double w = r == jb && in ? -bv : W[r];
                    T[tile_lower(c, r)][e] = have < 4 && q >= have ? old : w;
                }
            }
        }
    }
    if (!__builtin_constant_p(n)) settle<18>();
    return ok;
}

}  // namespace uqk
