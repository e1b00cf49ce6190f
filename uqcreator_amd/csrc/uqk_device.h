// uqk_device.h -- device-side closed forms shared by the closure and sweep
// kernels: entropy closures (U, DU), point fluxes, wave-level helpers.
// All arithmetic here is FP64.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "uqk.h"

namespace uqk {

struct ClosureParams {
    double gamma;      // positive adiabatic exponent
    double u_minus, u_plus;
    double g;
    double barrier;
    double alpha;
    double eps;
    int max_iter;
    int max_halvings;
    int du_exact;
    int safe;
};

struct ProblemParams {
    int problem;
    int flux;
    double cfl;
    double gamma;
    double g;
    double friction;
    int friction_dim;
};

template <int KIND> struct KindInfo;
template <> struct KindInfo<UQK_BOUNDED_BARRIER> { static constexpr int S = 1; };
template <> struct KindInfo<UQK_EULER1D> { static constexpr int S = 3; };
template <> struct KindInfo<UQK_EULER2D> { static constexpr int S = 4; };
template <> struct KindInfo<UQK_SHALLOW_WATER2D> { static constexpr int S = 3; };
template <> struct KindInfo<UQK_SHALLOW_WATER2D_BARRIER> { static constexpr int S = 3; };

// 1/h from v_rcp_f64 refined by two Newton steps
__device__ __forceinline__ double recip_f64(double h) {
    double r = __builtin_amdgcn_rcp(h);
    r = fma(r, fma(-h, r, 1.0), r);
    return fma(r, fma(-h, r, 1.0), r);
}

// ---------------------------------------------------------------------------
// Entropy closures.  U(Lambda) = (grad s)^{-1}(Lambda) per quadrature point.
// A division costs about 14 instructions, and the kernels that evaluate these
// are bound by the instructions they issue: the quotients of one argument
// share its reciprocal, and DU takes the density from U.
// ---------------------------------------------------------------------------

// Logistic map onto (u-, u+), evaluated on the branch whose exponential cannot
// overflow (boundedbarrier.cpp:19-31).
__device__ __forceinline__ double bb_u(double lam, double um, double up) {
    double ep = exp(lam);
    double en = 1.0 / ep;
    if (lam > 0.0) return up / (en + 1.0) + um * en / (1.0 + en);
    return um / (ep + 1.0) + up * ep / (1.0 + ep);
}

// d/dLambda of bb_u (boundedbarrier.cpp:67-80).
__device__ __forceinline__ double bb_du(double lam, double um, double up) {
    double ep = exp(lam);
    double en = 1.0 / ep;
    if (lam > 0.0) return en * (up - um) / (exp(-2.0 * lam) + 2.0 * en + 1.0);
    return ep * (up - um) / (1.0 + 2.0 * ep + exp(2.0 * lam));
}

// Density of the Euler closures from the duals (v0, v, w < 0), q = |v|^2, r =
// 1/w: exp((v0 - log(-w) - gamma - q / (2 w)) / (gamma - 1))
// (eulerclosure.cpp:7-12; eulerclosure2d.cpp:7-17, whose (-v4)^(1 / (1 - gamma))
// is taken into the exponential: equal up to rounding, no pow).
__device__ __forceinline__ double euler_rho(double v0, double q, double w, double r, double gm) {
#pragma clang fp contract(off)
    const double x = fma(-0.5 * q, r, (v0 - log(-w)) - gm), g1 = gm - 1.0, k = recip_f64(g1);
    const double e = x * k;
    // (the quotient corrected once: exp magnifies its error; an infinite one stays)
    return exp(__builtin_isfinite(e) ? fma(fma(-e, g1, x), k, e) : e);
}

// Vector form of U (the one Closure::Gradient uses).
template <int KIND>
__device__ __forceinline__ void closure_U(const ClosureParams& c, const double* L, double* out) {
    // (every fused multiply-add is written out: the residual checks and the
    // Newton kernels get the same bits)
#pragma clang fp contract(off)
    if constexpr (KIND == UQK_BOUNDED_BARRIER) {
        out[0] = bb_u(L[0], c.u_minus, c.u_plus);
    } else if constexpr (KIND == UQK_EULER1D) {
        // U = rho (1, -v/w, (v^2 - 2 w) / (2 w^2))
        const double r = recip_f64(L[2]), q = L[1] * L[1];
        const double rho = euler_rho(L[0], q, L[2], r, c.gamma);
        out[0] = rho;
        out[1] = -(L[1] * r) * rho;
        out[2] = (fma(0.5 * q, r, -1.0) * r) * rho;
    } else if constexpr (KIND == UQK_EULER2D) {
        const double r = recip_f64(L[3]), q = fma(L[1], L[1], L[2] * L[2]);
        const double rho = euler_rho(L[0], q, L[3], r, c.gamma);
        out[0] = rho;
        out[1] = -(L[1] * r) * rho;
        out[2] = -(L[2] * r) * rho;
        out[3] = (fma(0.5 * q, r, -1.0) * r) * rho;
    } else if constexpr (KIND == UQK_SHALLOW_WATER2D) {
        // shallowwaterclosure2d.cpp:10-14
        double c0 = fma(L[2], L[2], fma(L[1], L[1], 2.0 * L[0]));
        out[0] = 0.5 * c0 / c.g;
        out[1] = 0.5 * L[1] * c0 / c.g;
        out[2] = 0.5 * fma(L[2] * L[2], L[2], fma(L[1] * L[1], L[2], 2.0 * L[0] * L[2])) / c.g;
    } else {
        // entropy |q|^2/(2h) + g h^2/2 - eps log h: h solves g h - eps/h = c
        double cc = fma(0.5, fma(L[1], L[1], L[2] * L[2]), L[0]);
        double r = sqrt(fma(cc, cc, 4.0 * c.g * c.barrier));
        double h = cc > 0.0 ? (cc + r) / (2.0 * c.g) : (2.0 * c.barrier) / (r - cc);
        out[0] = h;
        out[1] = h * L[1];
        out[2] = h * L[2];
    }
}

// Matrix form of U (U(const Matrix&), used for uQ).  Only Euler2D differs:
// pow(-exp(a) v4, 1/(1+gamma)) (eulerclosure2d.cpp:19-32).
template <int KIND>
__device__ __forceinline__ void closure_U_mat(const ClosureParams& c, const double* L, double* out) {
    if constexpr (KIND == UQK_EULER2D) {
        const double gm = -c.gamma;
        double v1 = L[0], v2 = L[1], v3 = L[2], v4 = L[3];
        double e = pow(-exp((v2 * v2 + v3 * v3 - 2.0 * v1 * v4 - 2.0 * v4 * gm) / (2.0 * v4)) * v4, 1.0 / (1.0 + gm));
        out[0] = e;
        out[1] = -(v2 * e / v4);
        out[2] = -(v3 * e / v4);
        out[3] = -(e * (-v2 * v2 - v3 * v3 + 2.0 * v4)) / (2.0 * v4 * v4);
    } else {
        closure_U<KIND>(c, L, out);
    }
}

// Packed lower triangle of DU: entry p(l, m) = l*(l+1)/2 + m for m <= l holds
// dU_l/dLambda_m.  The Hessian's upper triangle only reads these
// (closure.cpp:265 with dposv 'U').  The Euler closures take U's density, rho.
template <int KIND>
__device__ __forceinline__ void closure_DU(const ClosureParams& c, const double* L, double rho, double* y) {
    if constexpr (KIND == UQK_BOUNDED_BARRIER) {
        y[0] = bb_du(L[0], c.u_minus, c.u_plus);
    } else if constexpr (KIND == UQK_EULER1D || KIND == UQK_EULER2D) {
        // U = rho f, f = (1, -v/w, h) with h = (q/(2w) - 1)/w = E/rho (total
        // energy over density); rho' = k rho f' with k = 1/(gamma - 1) and
        // f' = (1, -v/w, h') = d(log rho)/dLambda / k, h' = (q/(2w) - 1)/w
        // likewise; so DU = k rho f f^T + rho df/dLambda
        // (eulerclosure.cpp:37-56, eulerclosure2d.cpp:54-88)
        constexpr int D = KIND == UQK_EULER1D ? 1 : 2;
        const double w = L[D + 1], r = recip_f64(w), k = recip_f64(c.gamma - 1.0);
        double q = 0.0, m[D];  // m = -v/w, the velocity
#pragma unroll
        for (int i = 0; i < D; ++i) {
            m[i] = -(L[1 + i] * r);
            q += L[1 + i] * L[1 + i];
        }
        const double h = (0.5 * q * r - 1.0) * r, kr = k * rho, rr = rho * r;
        y[0] = kr;
#pragma unroll
        for (int i = 0; i < D; ++i) {
            const int l = 1 + i;
            y[l * (l + 1) / 2] = kr * m[i];
#pragma unroll
            for (int j = 0; j <= i; ++j) y[l * (l + 1) / 2 + 1 + j] = kr * m[i] * m[j] - (i == j ? rr : 0.0);
        }
        constexpr int e = D + 1, at = e * (e + 1) / 2;
        y[at] = kr * h;
#pragma unroll
        for (int j = 0; j < D; ++j) y[at + 1 + j] = kr * h * m[j] - rr * m[j];  // dh/dv = v/w^2 = -m/w
        // dh/dw = 1/w^2 - q/w^3
        if (KIND == UQK_EULER1D && !c.du_exact)
            y[at + e] = (L[1] * L[1] * (w * w * w) + r * r) * rho + kr * h * h;  // as shipped
        else
            y[at + e] = kr * h * h + rr * r * (1.0 - q * r);
    } else if constexpr (KIND == UQK_SHALLOW_WATER2D) {
        // shallowwaterclosure2d.cpp:39-49
        const double g = c.g;
        y[0] = 1.0 / g;
        y[1] = L[1] / g;
        y[2] = (L[0] + 1.5 * L[1] * L[1] + 0.5 * L[2] * L[2]) / g;
        y[3] = L[2] / g;
        y[4] = L[1] * L[2] / g;
        y[5] = 0.5 * (2.0 * L[0] + L[1] * L[1] + 3.0 * L[2] * L[2]) / g;
    } else {
        // DU = h' a a^T + h diag(0,1,1), a = (1, L1, L2), h' = dh/dc = h / r
        double cc = L[0] + 0.5 * (L[1] * L[1] + L[2] * L[2]);
        double r = sqrt(cc * cc + 4.0 * c.g * c.barrier);
        double h = cc > 0.0 ? (cc + r) / (2.0 * c.g) : (2.0 * c.barrier) / (r - cc);
        double hp = h / r;
        y[0] = hp;
        y[1] = hp * L[1];
        y[2] = hp * L[1] * L[1] + h;
        y[3] = hp * L[2];
        y[4] = hp * L[1] * L[2];
        y[5] = hp * L[2] * L[2] + h;
    }
}

// ---------------------------------------------------------------------------
// 1/x and sqrt(x) to an ulp: v_rcp_f64 with two Newton steps and v_rsq_f64
// with two of Goldschmidt's, in place of the correctly rounded divide and root,
// which take four times the instructions (and most of the time of the point
// fluxes).  Zero, infinities and NaN as 1/x and sqrt(x) have them.
__device__ __forceinline__ double recip_any(double x) {
    const double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    const double r1 = fma(r, e, r);
    e = fma(-x, r1, 1.0);
    const double r2 = fma(r1, e, r1);
    return __builtin_isfinite(r2) ? r2 : r;
}
__device__ __forceinline__ double sqrt_f64(double x) {
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r, h = 0.5 * r;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    g = fma(fma(-g, g, x), h, g);
    return x == 0.0 || x == __builtin_inf() ? x : g;
}

// Velocity, pressure and wave speed at a point (euler2d.cpp:88-112,
// shallowwater2d.cpp:21-65), what both sides of an edge bring into its flux.
struct PointState {
    double vx, vy, p, c;
};
template <int S> __device__ __forceinline__ PointState point_state(const ProblemParams& p, const double* u) {
#pragma clang fp contract(off)
    PointState q{0.0, 0.0, 0.0, 0.0};
    if constexpr (S >= 3) {
        const double ri = recip_any(u[0]);
        q.vx = u[1] * ri;
        q.vy = u[2] * ri;
        if constexpr (S == 4) {
            q.p = (p.gamma - 1.0) * fma(-0.5 * u[0], fma(q.vx, q.vx, q.vy * q.vy), u[3]);
            q.c = sqrt_f64(p.gamma * q.p * ri);
        } else {
            q.p = 0.5 * p.g * u[0] * u[0];
            q.c = sqrt_f64(p.g * u[0]);
        }
    }
    return q;
}

// Point fluxes G(u, v, nUnit, n): the outward flux of the cell holding u
// through an edge with unit normal nu and scaled normal n; a and b are the
// point_states of u and v.
// ---------------------------------------------------------------------------
template <int S>
__device__ __forceinline__ void point_flux(const ProblemParams& p, const double* u, const PointState& a,
                                           const double* v, const PointState& b, double nux, double nuy, double nx,
                                           double ny, double* out) {
    if (p.problem == UQK_BURGERS) {
        if (p.flux == UQK_FLUX_REFERENCE) {
            // burgers.cpp:21-28
            double w = (u[0] * nux > 0) ? u[0] : v[0];
            out[0] = 0.5 * w * w * nx;
        } else {
            // local Lax-Friedrichs (julia/Tensorization/IPMSolver.jl:39-42)
            double beta = fmax(fabs(u[0]), fabs(v[0]));
            out[0] = 0.5 * (0.5 * u[0] * u[0] + 0.5 * v[0] * v[0]) * nx - 0.5 * beta * (v[0] - u[0]) * fabs(nx);
        }
        return;
    }
    if constexpr (S >= 3) {
        // F . n = (rho un, q1 un + p nx, q2 un + p ny, (E + p) un), un the
        // velocity along the scaled normal (euler2d.cpp:95-112,
        // shallowwater2d.cpp:21-65); the reciprocals and square roots are
        // those of point_state, the cell's own once for all its edges
        const double nn = sqrt_f64(nx * nx + ny * ny);
        const double wu = a.vx * nx + a.vy * ny, wv = b.vx * nx + b.vy * ny;
        double Fu[S], Fv[S];
        Fu[0] = u[1] * nx + u[2] * ny;
        Fv[0] = v[1] * nx + v[2] * ny;
        Fu[1] = fma(u[1], wu, a.p * nx);
        Fv[1] = fma(v[1], wv, b.p * nx);
        Fu[2] = fma(u[2], wu, a.p * ny);
        Fv[2] = fma(v[2], wv, b.p * ny);
        if constexpr (S == 4) {
            Fu[3] = (u[3] + a.p) * wu;
            Fv[3] = (v[3] + b.p) * wv;
        }
        const double unu = nux * a.vx + nuy * a.vy, unv = nux * b.vx + nuy * b.vy;
        if (p.flux == UQK_FLUX_REFERENCE) {
            // HLL with Davis wave speeds (euler2d.cpp:52-87)
            const double lmin = unu - a.c, lmax = unv + b.c;
            const double f = recip_any(lmax - lmin), ll = lmax * lmin * nn;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const double h = f * ((lmax * Fu[s] - lmin * Fv[s]) + ll * (v[s] - u[s]));
                out[s] = lmin >= 0 ? Fu[s] : lmax <= 0 ? Fv[s] : h;
            }
        } else {
            const double smax = 0.5 * fmax(fabs(unu) + a.c, fabs(unv) + b.c) * nn;
#pragma unroll
            for (int s = 0; s < S; ++s) out[s] = 0.5 * (Fu[s] + Fv[s]) - smax * (v[s] - u[s]);
        }
    }
}

// Problem::ComputeDt for one quadrature point (burgers.cpp:114-122,
// euler2d.cpp:114-134; SW2D mirrors Euler2D with c = sqrt(g h)).
template <int S>
__device__ __forceinline__ double point_dt(const ProblemParams& p, const double* u, double dx) {
    if (p.problem == UQK_BURGERS) return p.cfl * dx / fabs(u[0]);
    if constexpr (S >= 3) {
        // min |1 / w| over the wave speeds w as 1 / max |w|: one reciprocal
        const PointState q = point_state<S>(p, u);
        return (p.cfl / dx) * recip_any(fmax(fmax(fabs(q.vy - q.c), fabs(q.vy + q.c)),
                                             fmax(fabs(q.vx + q.c), fabs(q.vx - q.c))));
    }
    return 1e10;
}

// ---------------------------------------------------------------------------
// Wave helpers (wave64).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_xor(v, off, 64));
    return v;
}

}  // namespace uqk
