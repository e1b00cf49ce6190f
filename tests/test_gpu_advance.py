"""The advance where its split over lanes changes: two points of a wavefront's
cells fewer or more than 32 and 64, more than two passes over the lanes, one
point, and one to four states; against the oracle, with wall cells on the rim."""
import numpy as np
import pytest

from test_gpu_sweeps import _oracle_closure, _oracle_mesh
from uqcreator_amd import mesh as meshes
from uqcreator_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q", [1, 2, 16, 31, 32, 33, 64, 65, 130])
@pytest.mark.parametrize("kind", [native.EULER2D, native.SHALLOW_WATER2D, native.BOUNDED_BARRIER])
def test_advance_over_points(oracle, kind, q):
    rng = np.random.default_rng(q)
    deg = min(q - 1, 17)  # past one tile of 16 moments
    b = native.Basis(1, [deg], q)
    kw, flux = {}, native.FLUX_REFERENCE
    if kind == native.BOUNDED_BARRIER:
        m = meshes.mesh1d(37, 0.0, 3.0)
        pk, base = native.BURGERS, np.array([6.0])
        kw = dict(u_minus=2.9, u_plus=12.1)
    elif kind == native.EULER2D:
        m = meshes.naca_ogrid(16, 5, radius=5.0, first_height=2e-2)
        pk, base = native.EULER2D_PROBLEM, np.array([1.0, 0.5, 0.1, 2.5])
    else:
        m = meshes.quad_grid(7, 9, -1, 1, -1, 1, native.BC_SWWALL)
        pk, base = native.SHALLOW_WATER2D_PROBLEM, np.array([1.5, 0.3, -0.2])
    print("case: advance kind", kind, "Q", b.Q, "M", b.M, "cells", m.n_cells, flush=True)
    S = native.STATES[kind]
    uq = base * (1 + 0.05 * rng.normal(size=(m.n_cells, b.Q, S)))
    u = np.ascontiguousarray(oracle.reconstruct(S, b.phiw, uq))
    prob = native.problem(pk, flux=flux, cfl=0.4)
    oprob = oracle.problem(pk, flux=flux, cfl=0.4)
    cl = native.GpuClosure(kind, b, **kw)
    du, duq = native.DeviceArray.from_host(u), native.DeviceArray.from_host(uq)
    dun = native.DeviceArray.from_host(np.zeros_like(u))
    dt = 1e-3
    cl.advance(prob, native.DeviceMesh(m), dt, du, duq, dun)
    want = oracle.advance(oprob, _oracle_mesh(oracle, m), b.phiw, b.xi, dt, u, uq)
    # sums of at most 4 Q fluxes, each to some ulps
    scale = np.maximum(np.abs(u).max(axis=(0, 1)), np.abs(want).max(axis=(0, 1)))
    assert (np.abs(dun.download() - want) / scale).max() < 1e-12
