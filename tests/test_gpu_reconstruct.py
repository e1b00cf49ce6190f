"""The moment reconstruction on both sides of the size at which it becomes a
matrix product, with cells of different orders, against the oracle."""
import numpy as np
import pytest

from uqcreator_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [native.BOUNDED_BARRIER, native.SHALLOW_WATER2D, native.EULER2D])
@pytest.mark.parametrize("degree,q", [(0, 1), (0, 31), (0, 32), (1, 2), (1, 15), (1, 16), (2, 10), (2, 11), (3, 7),
                                      (3, 8), (4, 6), (4, 7)])
def test_few_moments_and_points(oracle, kind, degree, q):
    b = native.Basis(1, list(range(degree + 1)), q)
    S = native.STATES[kind]
    rng = np.random.default_rng(100 * degree + q)
    for n in (1, 255, 4099):
        print("case: reconstruct S", S, "M", b.M, "Q", b.Q, "cells", n, flush=True)
        nt = rng.integers(1, b.M + 1, n).astype(np.int32)
        uq = rng.normal(0, 1, (n, b.Q, S))
        cl = native.GpuClosure(kind, b)
        duq, dnt = native.DeviceArray.from_host(uq), native.DeviceArray.from_host(nt)
        for order in (None, nt):
            u = native.DeviceArray.from_host(np.full((n, b.M, S), np.nan))
            cl.reconstruct(duq, u, nt_cell=None if order is None else dnt)
            want = oracle.reconstruct(S, b.phiw, uq, nt_cell=order)
            # sums of Q <= 32 products of size one, each rounded once
            np.testing.assert_allclose(u.download(), want, rtol=0, atol=32 * 2.3e-16 * np.abs(uq).max() *
                                       np.abs(b.phiw).sum(axis=0).max())
