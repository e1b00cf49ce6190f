"""One factored Newton step of every form of the register-tile factorisation,
against the oracle's: the direction has to be right to rounding times the
condition number.  (Converged duals do not show an error of 1e-8 in a step: the
iteration takes it out again.)  The forms that keep an inverse take exactly one
step because the tolerance lies between the norms before and after it; a second
time step, with other moments, then runs on what the first one kept."""
import numpy as np
import pytest

from test_gpu_tile import CASES as TILE_CASES
from test_gpu_tile import _cells
from test_gpu_wide import CASES as WIDE_CASES
from uqcreator_amd import mesh as meshes
from uqcreator_amd import native

pytestmark = pytest.mark.gpu

WAVE_CASES = [(native.BOUNDED_BARRIER, 1, [5], 12), (native.EULER1D, 2, [4], 7), (native.EULER2D, 2, [3], 5),
              (native.SHALLOW_WATER2D, 2, [3], 5), (native.SHALLOW_WATER2D_BARRIER, 2, [3], 5)]
# (a basis of one function or two varies too little for the bounds below)
TILE_CASES = [c for c in TILE_CASES if c[2][-1] > 1]


def _problem(oracle, kind, d, degrees, q1, n, alpha, seed):
    """Cells, a start at which the gradient's norm is about 1e-2, the oracle's
    next iterate, and the norms of both."""
    b = native.Basis(d, degrees, q1)
    rng = np.random.default_rng(seed)
    levels = np.asarray(b.ntotal_per_level, np.int32)
    nt = levels[rng.integers(0, len(levels), n)].astype(np.int32)
    c, u, lam_star, _, kw = _cells(oracle, kind, b, n, nt, rng)
    if kind == native.BOUNDED_BARRIER:
        kw = dict(u_minus=3.0, u_plus=12.0)
    c.alpha = alpha

    def norms(x):
        return np.array([np.linalg.norm(oracle.gradient(c, b.phi, b.phiw, np.ascontiguousarray(x[j]), u[j],
                                                        nt=int(nt[j]))) for j in range(n)])

    away = rng.uniform(-1, 1, lam_star.shape) * (np.arange(b.M)[None, :, None] < nt[:, None, None])
    if kind != native.BOUNDED_BARRIER:
        away *= lam_star  # (one relative change per dual: a temperature dual keeps its sign)
    lam0 = lam_star + 1e-4 * away
    lam0 = lam_star + 1e-4 * away * (1e-2 / norms(lam0))[:, None, None]
    c.max_iter = 1
    one = lam0.copy()
    st, _ = oracle.solve_closure(c, b.phi, b.phiw, u, one, nt_cell=nt)
    assert (st == 0).all()
    return b, kw, nt, u, lam_star, lam0, one, norms(lam0), norms(one)


def _check_step(lam, lam0, one, name):
    d, want = lam - lam0, one - lam0
    err = (np.abs(d - want).max(axis=(1, 2)) / np.abs(want).max(axis=(1, 2))).max()
    print("case: one step", name, "error", err, flush=True)
    # the gradient, 1e-2 of moments of order one, to 1e-14, times a condition below 1e5
    assert err < 1e-9


@pytest.mark.parametrize("form,case", [("wave", c) for c in WAVE_CASES] + [("tile", c) for c in TILE_CASES] +
                         [("wide", c) for c in WIDE_CASES])
def test_plain_step(oracle, form, case):
    kind, d, degrees, q1 = case
    n = 600 if kind == native.BOUNDED_BARRIER and form == "wide" else 67  # (more cells than workgroups)
    b, kw, nt, u, _, lam0, one, _, _ = _problem(oracle, kind, d, degrees, q1, n, 1.0, 51)
    cl = native.GpuClosure(kind, b, max_iterations=1, alpha=1.0, **kw)
    cl.set_kernel({"wave": native.KERNEL_WAVE, "tile": native.KERNEL_GENERIC, "wide": native.KERNEL_BLOCK}[form])
    lam = lam0.copy()
    cl.solve_host(u, lam, nt_cell=None if form == "wave" else nt)
    _check_step(lam, lam0, one, "%s kind %d n %d" % (form, kind, cl.S * b.M))


@pytest.mark.parametrize("case", WAVE_CASES)
def test_step_that_keeps_its_inverse_within_the_call(oracle, case):
    kind, d, degrees, q1 = case
    # (nearly undamped, so that one step ends below the tolerance; below 1, so
    # that the call keeps inverses)
    b, kw, nt, u, _, lam0, one, g0, g1 = _problem(oracle, kind, d, degrees, q1, 67, 0.99, 53)
    eps = np.sqrt(g0.min() * g1.max())
    assert g1.max() < 0.8 * eps and eps < 0.8 * g0.min()
    cl = native.GpuClosure(kind, b, epsilon=eps, alpha=0.99, precision=native.MIXED, **kw)
    cl.set_kernel(native.KERNEL_WAVE)
    lam = lam0.copy()
    st, it = cl.solve_host(u, lam)
    assert (st == 0).all() and (it == 1).all()
    _check_step(lam, lam0, one, "call, kind %d n %d" % (kind, cl.S * b.M))


@pytest.mark.parametrize("form,case", [("wave", c) for c in WAVE_CASES if c[0] != native.EULER1D] +
                         [("wide", c) for c in WIDE_CASES])
def test_step_that_keeps_its_inverse_across_steps(oracle, form, case):
    kind, d, degrees, q1 = case
    side = 25 if kind == native.BOUNDED_BARRIER and form == "wide" else 9
    n = side * side
    b, kw, nt, u, lam_star, lam0, one, g0, g1 = _problem(oracle, kind, d, degrees, q1, n, 1.0, 57)
    eps = np.sqrt(g0.min() * g1.max())
    assert g1.max() < 0.8 * eps and eps < 0.8 * g0.min()
    if kind == native.BOUNDED_BARRIER:
        m, pk = meshes.mesh1d(n, 0.0, 3.0), native.BURGERS
    else:
        m = meshes.quad_grid(side, side, -1, 1, -1, 1, native.BC_DIRICHLET)
        pk = native.EULER2D_PROBLEM if kind == native.EULER2D else native.SHALLOW_WATER2D_PROBLEM
    cl = native.GpuClosure(kind, b, epsilon=eps, alpha=1.0, precision=native.MIXED, **kw)
    cl.set_kernel(native.KERNEL_WAVE if form == "wave" else native.KERNEL_BLOCK)
    S = cl.S
    prob, dm = native.problem(pk, cfl=1e-6), native.DeviceMesh(m)
    du, dl = native.DeviceArray.from_host(u), native.DeviceArray.from_host(lam0)
    uq, us = native.DeviceArray((n, b.Q, S)), native.DeviceArray((n, b.M, S))
    st, it = native.DeviceArray(n, np.int32), native.DeviceArray(n, np.int32)
    dnt = None if form == "wave" else native.DeviceArray.from_host(nt)
    cl.step(prob, dm, du, dl, uq, us, st, it, nt_cell=dnt)
    assert (st.download() == 0).all() and (it.download() == 1).all()
    lam = dl.download()
    _check_step(lam, lam0, one, "%s, time loop, kind %d n %d" % (form, kind, S * b.M))
    # other moments, as far away on the other side: the kept inverses take over
    c = oracle.closure({native.BOUNDED_BARRIER: oracle.BB, native.EULER1D: oracle.EULER1D,
                        native.EULER2D: oracle.EULER2D, native.SHALLOW_WATER2D: oracle.SW2D,
                        native.SHALLOW_WATER2D_BARRIER: oracle.SW2D_BARRIER}[kind], eps=eps, du_exact=1, alpha=1.0,
                       **{k: v for k, v in kw.items() if k in ("barrier", "u_minus", "u_plus")})
    other = 2 * lam_star - lam0
    u2 = oracle.reconstruct(S, b.phiw, np.ascontiguousarray(oracle.eval_uq(c, b.phi, other, nt_cell=nt)), nt_cell=nt)
    du.upload(u2)
    cl.step(prob, dm, du, dl, uq, us, st, it, nt_cell=dnt)
    factors, kept = cl.last_closure_factorizations()
    print("case: second step", form, "kind", kind, "factorisations", factors, "kept steps", kept, flush=True)
    assert (st.download() == 0).all() and kept > 0.9 * n and factors < 0.1 * n
    lam = dl.download()
    for j in range(n):
        assert not lam[j, nt[j]:].any()
        g = oracle.gradient(c, b.phi, b.phiw, np.ascontiguousarray(lam[j]), u2[j], nt=int(nt[j]))
        assert np.linalg.norm(g) < eps * (1 + 1e-9) + 1e-13 * np.abs(u2[j]).max(), j
