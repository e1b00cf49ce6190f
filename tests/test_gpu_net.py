"""The fused network against the oracle and against itself: one row, the edges
of its 16- and 64-row workgroups, hidden widths that leave a wavefront fewer
than four tiles or none, and both row counts per workgroup, whose outputs agree
bit for bit."""
import numpy as np
import pytest

from test_gpu_mlp import _closure_c2, _random_params, _rel
from uqcreator_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [32, 96, 256, 320])
def test_rows_and_widths(oracle, hidden):
    b, cl = _closure_c2()
    net = native.WarmStartNet(cl, hidden=hidden, seed=3)
    dims = net.dims
    rng = np.random.default_rng(hidden)
    params = _random_params(dims, rng)
    net.set_params(params)
    rows = 4096 + 65  # above 4096 rows a workgroup takes 64 of them
    x = np.zeros((rows, dims[0]), np.float32)
    x[:, :45] = rng.normal(0, 1, (rows, 45))
    y = net.forward(native.DeviceArray.from_host(x)).download()
    want = oracle.mlp_forward(dims, params.astype(np.float64), x[-65:].astype(np.float64), emulate_bf16=True)
    # FP32 accumulation order and the BF16 roundings it flips, as in
    # test_forward_and_gradient_match_oracle
    err = _rel(y[-65:], want)
    print("case: fused network hidden", hidden, "error", err, flush=True)
    assert err < 5e-3
    for part in (1, 15, 16, 17, 63, 64, 65, 4096):
        z = net.forward(native.DeviceArray.from_host(np.ascontiguousarray(x[:part]))).download()
        np.testing.assert_array_equal(z, y[:part])
