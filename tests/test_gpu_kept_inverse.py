"""The kept inverses of the mixed time loop hold what a step stored and nothing
else: what the memory of their slots held before must not reach a result."""
import numpy as np
import pytest

from uqcreator_amd import native, solver, workloads

pytestmark = pytest.mark.gpu


def _burgers(cells):
    # 6 duals: a row of the inverse is padded to 8 entries
    b, m, u, lam = workloads.burgers_c1(cells)
    return (native.BOUNDED_BARRIER, dict(u_minus=2.9, u_plus=12.1, epsilon=1e-6), b, m, u, lam,
            native.problem(native.BURGERS, flux=native.FLUX_LAX_FRIEDRICHS, cfl=0.5))


def _shallow(cells, kind):
    # 30 duals: padded to 32
    from uqcreator_amd import mesh as meshes

    b = native.Basis(2, [3], 5)
    m = meshes.quad_grid(cells, cells, -1.0, 1.0, -1.0, 1.0, native.BC_DIRICHLET)
    u = workloads.project_ic(workloads.sw2d_dambreak_ic(), m.center, b)
    lam = np.zeros_like(u)
    lam[:, 0, 0] = 9.81 * u[:, 0, 0]
    kw = dict(epsilon=1e-7)
    if kind == native.SHALLOW_WATER2D_BARRIER:
        kw["barrier"] = 0.01
    return kind, kw, b, m, u, lam, native.problem(native.SHALLOW_WATER2D_PROBLEM, flux=native.FLUX_LAX_FRIEDRICHS,
                                                  cfl=0.4)


@pytest.mark.parametrize("case", ["burgers", "shallow", "shallow_barrier"])
def test_slots_may_have_held_nan(case):
    """The same loop with slots in memory that held NaN and in memory that held
    zeros: equal to the last bit, steps on kept inverses included.  (The
    allocator hands freed blocks of the slots' size out again.)"""
    kind, kw, b, m, u, lam, prob = (_burgers(300) if case == "burgers" else
                                    _shallow(16, native.SHALLOW_WATER2D if case == "shallow" else
                                             native.SHALLOW_WATER2D_BARRIER))
    n = native.STATES[kind] * b.M
    floats = m.n_cells * n * ((n + 3) // 4 * 4)
    out = []
    for value in (0.0, np.nan):
        print("case: kept inverses in recycled memory", case, "value", value, flush=True)
        cl = native.GpuClosure(kind, b, precision=native.MIXED, **kw)
        s = solver.GpuMomentSolver(cl, prob, m)
        s.set_state(u, lam)
        blocks = [native.DeviceArray.from_host(np.full(floats, value, np.float32)) for _ in range(8)]
        for x in blocks:
            x.free()
        s.run_device(1e3, max_steps=12)
        assert cl.last_kernel() == native.KERNEL_WAVE
        out.append((s.u.download(), s.lam.download(), s.newton_steps, cl.last_closure_factorizations()))
    assert out[0][3][1] > 0  # some steps ran on kept inverses
    assert out[0][2:] == out[1][2:]
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
