"""A Newton trial whose state overflows at one quadrature point has an infinite
gradient, and the line search halves the step (closure.cpp:159-184 compares
norms, and infinity is larger).  Kernels that take points in groups fill the
last group up: the fill must not turn that infinity into a NaN, which the
search would accept and end the cell on."""
import numpy as np
import pytest

from uqcreator_amd import native

pytestmark = pytest.mark.gpu

# (closure, uncertain dimensions, degrees, points per dimension, kernel)
CASES = [
    (native.EULER1D, 2, [4], 7, native.KERNEL_WAVE), (native.EULER2D, 2, [3], 5, native.KERNEL_WAVE),
    (native.EULER2D, 2, [2], 5, native.KERNEL_GENERIC), (native.EULER1D, 1, [5], 9, native.KERNEL_GENERIC),
    (native.EULER2D, 1, [2], 4, native.KERNEL_GENERIC), (native.EULER1D, 1, [3], 5, native.KERNEL_GENERIC),
    (native.EULER2D, 2, [5], 7, native.KERNEL_BLOCK), (native.EULER1D, 2, [6], 9, native.KERNEL_BLOCK),
    (native.EULER2D, 1, [15], 18, native.KERNEL_BLOCK),
]


def _cells(oracle, kind, b, n, rng):
    """(u, lambda) of n cells whose first Newton trial brings the temperature
    dual next to zero, and the density to infinity, at the last point alone:
    the moments are chosen for that trial, u = <U(lambda)> - H d."""
    S = native.STATES[kind]
    c = oracle.closure(oracle.EULER1D if kind == native.EULER1D else oracle.EULER2D, eps=1e-10, du_exact=1)
    us, lams = [], []
    for _ in range(100 * n):
        rho, p, v = rng.uniform(0.5, 2), rng.uniform(0.5, 2), rng.uniform(0.3, 1, S - 2)
        lam = np.zeros((b.M, S))
        lam[0] = oracle.DS(c, np.r_[rho, rho * v, p / 0.4 + 0.5 * rho * (v * v).sum()])
        lam[1:] = rng.normal(0, 0.01, (b.M - 1, S)) * np.abs(lam[0])
        at = b.phi @ lam
        trial = lam.copy()
        last = b.phi[-1]
        trial[:, -1] -= last / (last @ last) * (at[-1, -1] + 10.0 ** rng.uniform(-5, -4))
        if (at[:, -1] > -0.1).any() or ((b.phi @ trial)[:-1, -1] > -1e-2).any():
            continue
        H = oracle.hessian(c, b.phi, b.phiw, lam)
        H = np.triu(H) + np.triu(H, 1).T
        d = ((lam - trial) / c.alpha).T.reshape(-1)
        u = b.phiw.T @ np.array([oracle.U(c, x) for x in at]) - (H @ d).reshape(S, b.M).T
        # what the solver's own first trial gives
        d = np.linalg.solve(H, oracle.gradient(c, b.phi, b.phiw, lam, u)).reshape(S, b.M).T
        with np.errstate(over="ignore"):
            U = np.array([oracle.U(c, x) for x in b.phi @ (lam - c.alpha * d)])
        if np.isinf(U[-1]).all() and np.isfinite(U[:-1]).all():
            us.append(u)
            lams.append(lam)
        if len(us) == n:
            return c, np.ascontiguousarray(us), np.ascontiguousarray(lams)
    raise AssertionError("no such cells")


@pytest.mark.parametrize("precision", [native.FP64, native.MIXED])
@pytest.mark.parametrize("kind,d,degrees,q1,kernel", CASES)
def test_overflow_at_the_last_point_halves_the_step(oracle, kind, d, degrees, q1, kernel, precision):
    b = native.Basis(d, degrees, q1)
    c, u, lam0 = _cells(oracle, kind, b, 24, np.random.default_rng(37))
    lam_o = lam0.copy()
    st_o, it_o = oracle.solve_closure(c, b.phi, b.phiw, u, lam_o)
    print("case: overflow kind", kind, "M", b.M, "Q", b.Q, "kernel", kernel, "oracle", st_o.tolist(), flush=True)
    assert (st_o == 0).sum() >= 20
    cl = native.GpuClosure(kind, b, epsilon=1e-10, precision=precision)
    cl.set_kernel(kernel)
    lam = lam0.copy()
    st, it = cl.solve_host(u, lam)
    assert cl.last_kernel() == kernel
    np.testing.assert_array_equal(st, st_o)
    for j in np.flatnonzero(st == 0):
        g = oracle.gradient(c, b.phi, b.phiw, lam[j], u[j])
        # the kernel's ||grad L|| < 1e-10 to the rounding of its Q-term sums
        assert np.linalg.norm(g) < 1e-10 + 1e-13 * np.abs(u[j]).max(), j


@pytest.mark.parametrize("kind", [native.EULER1D, native.EULER2D])
def test_density_of_an_infinite_exponent(oracle, kind):
    """|v|^2 past the largest double: the density is infinite, as the
    reference's exponential gives it, not NaN."""
    b = native.Basis(1, [0], 1)
    S = native.STATES[kind]
    c = oracle.closure(oracle.EULER1D if kind == native.EULER1D else oracle.EULER2D)
    lam = np.full((8, 1, S), 0.5)
    lam[:, 0, -1] = -1.0
    lam[:, 0, 1] = [1e150, 1e153, 1.4e154, 1e155, 1e160, -1e170, 1e200, -1e300]
    with np.errstate(over="ignore", invalid="ignore"):
        want = oracle.mean_var(c, b.phi, b.phiw, lam)[:, :S]
    print("case: infinite exponent kind", kind, want.tolist(), flush=True)
    assert np.isinf(want).all()
    cl = native.GpuClosure(kind, b)
    mv = native.DeviceArray((8, 2 * S))
    cl.mean_var(native.DeviceArray.from_host(lam), mv)
    np.testing.assert_array_equal(mv.download()[:, :S], want)
