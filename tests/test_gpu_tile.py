"""The runtime-sized closure kernel (systems of fewer than 64 duals in register
tiles of 16 rows) against the FP64 oracle where its sizes can go wrong: one
row more or less than a tile, orders that are no multiple of the four pivots
of a step, the smallest and largest systems, more points than lanes, and cells
of different orders side by side."""
import numpy as np
import pytest

from uqcreator_amd import native

pytestmark = pytest.mark.gpu

# (closure, uncertain dimensions, degrees, points per dimension)
CASES = [
    (native.BOUNDED_BARRIER, 1, [0], 2), (native.BOUNDED_BARRIER, 1, [2], 4), (native.BOUNDED_BARRIER, 1, [14], 17),
    (native.BOUNDED_BARRIER, 1, [15], 18), (native.BOUNDED_BARRIER, 1, [16], 19),
    (native.BOUNDED_BARRIER, 1, [31], 34), (native.BOUNDED_BARRIER, 1, [46], 49),
    (native.BOUNDED_BARRIER, 1, [47], 64), (native.BOUNDED_BARRIER, 1, [62], 65),
    (native.EULER1D, 2, [1, 2, 3, 4, 5], 7), (native.EULER1D, 2, [5], 9),
    (native.EULER2D, 2, [1, 2, 3, 4], 6), (native.EULER2D, 2, [2], 4),
    (native.SHALLOW_WATER2D, 2, [1, 2, 3, 4], 5), (native.SHALLOW_WATER2D_BARRIER, 3, [1, 2], 5),
]


def _cells(oracle, kind, b, n, nt, rng):
    kw = dict(barrier=0.01) if kind == native.SHALLOW_WATER2D_BARRIER else {}
    names = {native.BOUNDED_BARRIER: "BB", native.EULER1D: "EULER1D", native.EULER2D: "EULER2D",
             native.SHALLOW_WATER2D: "SW2D", native.SHALLOW_WATER2D_BARRIER: "SW2D_BARRIER"}
    c = oracle.closure(getattr(oracle, names[kind]), eps=1e-10, du_exact=1, safe=1, **kw)
    lam = np.zeros((n, b.M, c.S))
    for j in range(n):
        m = nt[j]
        if kind == native.BOUNDED_BARRIER:
            lam[j, :m, 0] = rng.normal(0, 0.3, m) / (1 + np.arange(m))
            continue
        if kind == native.EULER1D:
            rho, v, p = rng.uniform(0.5, 2), rng.uniform(-1, 1), rng.uniform(0.5, 2)
            cons = np.array([rho, rho * v, p / 0.4 + 0.5 * rho * v * v])
        elif kind == native.EULER2D:
            rho, vx, vy, p = rng.uniform(0.5, 2), rng.uniform(-1, 1), rng.uniform(-1, 1), rng.uniform(0.5, 2)
            cons = np.array([rho, rho * vx, rho * vy, p / 0.4 + 0.5 * rho * (vx * vx + vy * vy)])
        else:
            h, vx, vy = rng.uniform(1, 3), rng.uniform(-1, 1), rng.uniform(-1, 1)
            cons = np.array([h, h * vx, h * vy])
        lam[j, 0] = oracle.DS(c, cons)
        lam[j, 1:m] = rng.normal(0, 0.01, (m - 1, c.S)) * np.abs(lam[j, 0])
    uq = np.ascontiguousarray(oracle.eval_uq(c, b.phi, lam, nt_cell=nt))
    u = oracle.reconstruct(c.S, b.phiw, uq, nt_cell=nt)
    lam0 = np.zeros_like(lam)
    if kind != native.BOUNDED_BARRIER:
        for j in range(n):
            lam0[j, 0] = oracle.DS(c, u[j, 0])
    return c, u, lam, lam0, kw


@pytest.mark.parametrize("kind,d,degrees,q1", CASES)
def test_closure_at_tile_edges(oracle, kind, d, degrees, q1):
    b = native.Basis(d, degrees, q1)
    rng = np.random.default_rng(17)
    n = 203
    levels = np.asarray(b.ntotal_per_level, np.int32)
    nt = levels[rng.integers(0, len(levels), n)].astype(np.int32)
    c, u, lam_star, lam0, kw = _cells(oracle, kind, b, n, nt, rng)
    if kind == native.BOUNDED_BARRIER:
        kw = dict(u_minus=3.0, u_plus=12.0)
    print("case: tiles kind", kind, "M", b.M, "Q", b.Q, "orders", levels.tolist(), flush=True)
    cl = native.GpuClosure(kind, b, epsilon=1e-10, safe_line_search=1, **kw)
    cl.set_kernel(native.KERNEL_GENERIC)
    lam = lam0.copy()
    st, it = cl.solve_host(u, lam, nt_cell=nt)
    assert cl.last_kernel() == native.KERNEL_GENERIC
    lam_o = lam0.copy()
    st_o, it_o = oracle.solve_closure(c, b.phi, b.phiw, u, lam_o, nt_cell=nt)
    np.testing.assert_array_equal(st, st_o)
    assert (st == 0).all()
    assert np.abs(it - it_o).max() <= 1
    # ||grad L|| < 1e-10 at both: duals equal to that over the smallest
    # curvature, which the cells keep above 1e-2
    scale = np.abs(lam_star).max(axis=(1, 2), keepdims=True)
    assert (np.abs(lam - lam_o) / np.maximum(scale, 1e-2)).max() < 1e-6
    assert (np.abs(lam - lam_star) / np.maximum(scale, 1e-2)).max() < 1e-6
    for j in range(n):
        assert not lam[j, nt[j]:].any()
        g = oracle.gradient(c, b.phi, b.phiw, np.ascontiguousarray(lam[j]), u[j], nt=int(nt[j]))
        assert np.linalg.norm(g) < 2e-10, j
