"""A run in several calls ends where one call ends, bit for bit: a call's first
step takes the full residual check, whose U, ComputeDt and moments have to be
those that the Newton kernel leaves to the later steps."""
import numpy as np
import pytest

from uqcreator_amd import mesh as meshes
from uqcreator_amd import native, solver, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [native.FP64, native.MIXED])
@pytest.mark.parametrize("chunk", [7, 20])
def test_euler2d_run_in_chunks(precision, chunk):
    b = native.Basis(2, [3], 5)
    m = meshes.naca_ogrid(128, 32)
    u0 = workloads.project_ic(workloads.euler2d_freestream_ic(), m.center, b)
    lam0 = np.zeros_like(u0)
    lam0[:, 0] = workloads.euler2d_ds(u0[:, 0])
    prob = native.problem(native.EULER2D_PROBLEM, flux=native.FLUX_LAX_FRIEDRICHS, cfl=0.4)
    out = []
    for step in (60, chunk):
        print("case: run in chunks of", step, "precision", precision, flush=True)
        cl = native.GpuClosure(native.EULER2D, b, epsilon=1e-6, precision=precision)
        s = solver.GpuMomentSolver(cl, prob, m)
        s.set_state(u0, lam0)
        while s.steps < 60:
            s.run_device(1e3, max_steps=min(step, 60 - s.steps))
        out.append((s.u.download(), s.lam.download(), s.t))
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
