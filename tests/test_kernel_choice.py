"""Which kernel takes a large system: the rule is host arithmetic on the LDS
that a workgroup needs, asked of the library itself."""
import ctypes

import numpy as np
import pytest

from uqcreator_amd import mesh as meshes
from uqcreator_amd import native, solver, workloads

LDS, CUS = 160 * 1024, 256


def _wide_takes(S, M, Q, cells=100000):
    # uqk::newton_wide_takes(int, int, int, int, int, long)
    f = getattr(native.lib(), "_ZN3uqk17newton_wide_takesEiiiiil")
    f.restype = ctypes.c_bool
    return f(S, M, Q, LDS, CUS, ctypes.c_long(cells))


@pytest.mark.parametrize("S,M,Q,takes", [
    (3, 35, 125, True), (3, 35, 190, True),     # four and two wavefronts in LDS
    (3, 35, 205, False), (3, 35, 216, False),   # one, beside two resident workgroups
    (3, 35, 245, False),                        # none
    (4, 24, 216, True), (4, 24, 230, False),
    (4, 28, 256, True), (4, 31, 216, True),     # one, beside one resident workgroup
    (4, 21, 300, True),                         # one, and more points than the workgroup kernel takes
    (3, 37, 40, True), (3, 38, 40, False), (4, 31, 40, True), (4, 32, 40, False),  # 111 and 127 duals
])
def test_wide_kernel(S, M, Q, takes):
    assert _wide_takes(S, M, Q) == takes


@pytest.mark.parametrize("S,M,Q,cells,takes", [
    (1, 64, 66, 1, False), (1, 64, 66, 512, False), (1, 64, 66, 513, True),  # two workgroups resident
    (1, 76, 78, 512, False), (1, 76, 78, 513, True), (4, 16, 40, 1, True), (3, 35, 125, 1, True),
])
def test_wide_kernel_for_few_cells(S, M, Q, cells, takes):
    assert _wide_takes(S, M, Q, cells) == takes


@pytest.mark.parametrize("S,M,tile_rows", [(4, 16, 4), (3, 22, 5), (4, 24, 6), (3, 35, 7), (4, 28, 7), (4, 31, 8)])
def test_kept_inverse_takes_the_tiles_of_its_rows(S, M, tile_rows):
    f = getattr(native.lib(), "_ZN3uqk23newton_wide_kept_floatsEii")  # uqk::newton_wide_kept_floats(int, int)
    f.restype = ctypes.c_long
    assert f(S, M) == 256 * (tile_rows * (tile_rows + 1) // 2)


@pytest.mark.gpu
def test_slots_follow_the_number_of_cells():
    """One context that runs many cells, few and many again: what the kernel of
    one size keeps of a cell's factorisation is not read by that of the other."""
    b = native.Basis(1, [63], 66)
    prob = native.problem(native.BURGERS, flux=native.FLUX_LAX_FRIEDRICHS, cfl=0.5)
    kw = dict(u_minus=2.9, u_plus=12.1, epsilon=1e-6, precision=native.MIXED)

    def run(cl, cells):
        print("case: 64 duals, one state,", cells, "cells", flush=True)
        m = meshes.mesh1d(cells, 0.0, 3.0)
        u = workloads.project_ic(workloads.burgers_step_ic(), m.center, b)
        u[:, 1:] *= 0.1
        s = solver.GpuMomentSolver(cl, prob, m)
        s.set_state(u, np.zeros_like(u))
        s.run_device(1e3, max_steps=6)
        assert (s.status.download() == 0).all()
        return s.u.download(), s.lam.download(), s.newton_steps, cl.last_closure_factorizations()

    one = native.GpuClosure(native.BOUNDED_BARRIER, b, **kw)
    for cells in (700, 300, 700):
        got, want = run(one, cells), run(native.GpuClosure(native.BOUNDED_BARRIER, b, **kw), cells)
        assert got[2:] == want[2:] and got[3][1] > 0
        np.testing.assert_array_equal(got[0], want[0])
        np.testing.assert_array_equal(got[1], want[1])


@pytest.mark.gpu
def test_wave_count_is_the_wave_kernels():
    """The launch shape's number of wavefronts is the wave kernel's: set before
    (a tuned context, say), it does not idle the large systems' SIMDs."""
    b = native.Basis(3, [4], 5)
    rng = np.random.default_rng(47)
    n = 4096
    h, vx, vy = rng.uniform(1, 3, n), rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    lam = np.zeros((n, b.M, 3))
    lam[:, 0] = np.stack([9.81 * h - 0.5 * (vx * vx + vy * vy), vx, vy], -1)
    lam[:, 1:] = rng.normal(0, 0.01, (n, b.M - 1, 3)) * np.abs(lam[:, :1])
    cl = native.GpuClosure(native.SHALLOW_WATER2D_BARRIER, b, epsilon=1e-8, barrier=0.01, safe_line_search=1)
    dl, uq, u = native.DeviceArray.from_host(lam), native.DeviceArray((n, b.Q, 3)), native.DeviceArray((n, b.M, 3))
    cl.eval_uq(dl, uq)
    cl.reconstruct(uq, u)
    lam[:, 1:] = 0.0
    times = {}
    for waves in (0, 1):
        cl.set_launch_shape(waves, 0)
        for _ in range(4):
            x = native.DeviceArray.from_host(lam)
            assert cl.solve(u, x) == 0 and cl.last_kernel() == native.KERNEL_BLOCK
            times[waves] = min(times.get(waves, np.inf), cl.last_closure_ms())
    print("case: 105 duals, launch shape of one wavefront", times, flush=True)
    # equal work; the tables leave LDS for one workgroup, whose one wavefront
    # would take three to four times as long
    assert times[1] < 1.5 * times[0]
