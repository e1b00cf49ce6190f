"""The workgroup-per-cell closure kernel at the sizes that are its own: 128
duals, 112 to 127 of fewer than four states, and tables of which LDS holds one
wavefront's or none; FP64, the FP32 Hessian of the mixed closure and the kept
FP32 factors of its time loop, against the FP64 oracle."""
import numpy as np
import pytest

from test_gpu_tile import _cells
from test_kernel_choice import _wide_takes
from uqcreator_amd import native, solver, workloads

pytestmark = pytest.mark.gpu

# (closure, uncertain dimensions, degrees, points per dimension)
CASES = [
    (native.EULER2D, 1, [31], 34), (native.EULER2D, 1, [9, 20, 31], 36),  # 128 duals
    (native.EULER1D, 1, [37], 40), (native.SHALLOW_WATER2D, 1, [10, 41], 44), (native.BOUNDED_BARRIER, 1, [127], 130),
    (native.SHALLOW_WATER2D_BARRIER, 3, [1, 4], 6),  # 105 duals, 216 points
    (native.EULER2D, 1, [20], 256),                  # 84 duals, the most points
]


def _context(oracle, kind, d, degrees, q1, n, seed):
    b = native.Basis(d, degrees, q1)
    assert not _wide_takes(native.STATES[kind], b.M, b.Q, n)
    rng = np.random.default_rng(seed)
    levels = np.asarray(b.ntotal_per_level, np.int32)
    nt = levels[rng.integers(0, len(levels), n)].astype(np.int32)
    c, u, lam_star, lam0, kw = _cells(oracle, kind, b, n, nt, rng)
    if kind == native.BOUNDED_BARRIER:
        kw = dict(u_minus=3.0, u_plus=12.0)
    return b, c, nt, u, lam_star, lam0, kw


@pytest.mark.parametrize("precision", [native.FP64, native.MIXED])
@pytest.mark.parametrize("kind,d,degrees,q1", CASES)
def test_closure(oracle, kind, d, degrees, q1, precision):
    n = 97
    b, c, nt, u, lam_star, lam0, kw = _context(oracle, kind, d, degrees, q1, n, 61)
    print("case: workgroup kind", kind, "M", b.M, "Q", b.Q, "precision", precision, flush=True)
    cl = native.GpuClosure(kind, b, epsilon=1e-10, safe_line_search=1, precision=precision, **kw)
    lam = lam0.copy()
    st, it = cl.solve_host(u, lam, nt_cell=nt)
    assert cl.last_kernel() == native.KERNEL_BLOCK
    lam_o = lam0.copy()
    st_o, it_o = oracle.solve_closure(c, b.phi, b.phiw, u, lam_o, nt_cell=nt)
    np.testing.assert_array_equal(st, st_o)
    assert (st == 0).all()
    # (the FP32 Hessian changes the path a little, not where it ends)
    assert np.abs(it - it_o).max() <= 1 if precision == native.FP64 else it.mean() <= it_o.mean() + 1
    # ||grad L|| < 1e-10 at both: duals equal to that over the smallest
    # curvature, which the cells keep above 1e-2
    scale = np.abs(lam_star).max(axis=(1, 2), keepdims=True)
    assert (np.abs(lam - lam_o) / np.maximum(scale, 1e-2)).max() < 1e-6


@pytest.mark.parametrize("kind,d,degrees,q1", CASES)
def test_one_step(oracle, kind, d, degrees, q1):
    n = 67
    b, c, nt, u, lam_star, lam0, kw = _context(oracle, kind, d, degrees, q1, n, 63)
    c.max_iter = 1
    cl = native.GpuClosure(kind, b, max_iterations=1, safe_line_search=1, **kw)
    lam, lam_o = lam0.copy(), lam0.copy()
    cl.solve_host(u, lam, nt_cell=nt)
    assert cl.last_kernel() == native.KERNEL_BLOCK
    oracle.solve_closure(c, b.phi, b.phiw, u, lam_o, nt_cell=nt)
    scale = np.maximum(np.abs(lam_star).max(axis=(1, 2), keepdims=True), 1e-2)
    err = (np.abs(lam - lam_o) / scale).max()
    print("case: workgroup one step kind", kind, "n", c.S * b.M, "error", err, flush=True)
    assert err < 1e-10  # rounding times a condition below 1e5


@pytest.mark.parametrize("case", ["euler2d_128", "dambreak_216_points", "euler2d_128_orders"])
def test_time_loop_keeps_factors(case):
    """The mixed loop on kept factors ends where the FP64 loop ends (both to
    ||grad L|| below the workload's tolerance)."""
    nt = None
    if case.startswith("euler2d"):
        b = native.Basis(1, [9, 20, 31] if case.endswith("orders") else [31], 34)
        _, m, _, _, _ = workloads.euler2d_c4(64, 16)
        u = workloads.project_ic(workloads.euler2d_freestream_ic(), m.center, b)
        if case.endswith("orders"):
            levels = np.asarray(b.ntotal_per_level, np.int32)
            nt = levels[np.random.default_rng(67).integers(0, 3, m.n_cells)].astype(np.int32)
            u *= (np.arange(b.M)[None, :, None] < nt[:, None, None])
        lam = np.zeros_like(u)
        lam[:, 0] = workloads.euler2d_ds(u[:, 0])
        kind, kw, eps = native.EULER2D, {}, 1e-6
        prob = native.problem(native.EULER2D_PROBLEM, flux=native.FLUX_LAX_FRIEDRICHS, cfl=0.4)
    else:
        b, m, u = workloads.sw2d_c5(32, 4, 6)
        lam = np.zeros_like(u)
        lam[:, 0, 0] = 9.81 * u[:, 0, 0]
        kind, kw, eps = native.SHALLOW_WATER2D_BARRIER, dict(barrier=0.01), 1e-8
        prob = native.problem(native.SHALLOW_WATER2D_PROBLEM, flux=native.FLUX_LAX_FRIEDRICHS, cfl=0.4)
    assert not _wide_takes(native.STATES[kind], b.M, b.Q, m.n_cells)
    out = []
    for precision in (native.FP64, native.MIXED):
        print("case: workgroup loop", case, "precision", precision, flush=True)
        cl = native.GpuClosure(kind, b, epsilon=eps, precision=precision, **kw)
        s = solver.GpuMomentSolver(cl, prob, m, nt_cell=nt)
        s.set_state(u, lam)
        s.run_device(1e3, max_steps=6)
        assert cl.last_kernel() == native.KERNEL_BLOCK
        assert (s.status.download() == 0).all()
        out.append(s.u.download())
        if precision == native.MIXED:
            assert cl.last_closure_factorizations()[1] > 0
    ref, got = out
    assert np.abs(got - ref).max() / np.abs(ref).max() < 1e-7
