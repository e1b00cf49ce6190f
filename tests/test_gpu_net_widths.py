"""The network where its width and rows choose between the fused kernel and one
GEMM per layer: both give the same bits."""
import numpy as np
import pytest

from test_gpu_mlp import _closure_c2, _random_params, _rel
from uqcreator_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [288, 320, 416, 448])
def test_rows_around_the_choice(oracle, hidden):
    b, cl = _closure_c2()
    net = native.WarmStartNet(cl, hidden=hidden, seed=3)
    dims = net.dims
    rng = np.random.default_rng(hidden)
    params = _random_params(dims, rng)
    net.set_params(params)
    x = np.zeros((130, dims[0]), np.float32)
    x[:, :45] = rng.normal(0, 1, (130, 45))
    y = net.forward(native.DeviceArray.from_host(x)).download()
    want = oracle.mlp_forward(dims, params.astype(np.float64), x.astype(np.float64), emulate_bf16=True)
    err = _rel(y, want)
    print("case: network width", hidden, "error", err, flush=True)
    # FP32 accumulation order and the BF16 roundings it flips, as in
    # test_forward_and_gradient_match_oracle
    assert err < 5e-3
    for part in (1, 15, 16, 17, 33):
        z = net.forward(native.DeviceArray.from_host(np.ascontiguousarray(x[:part]))).download()
        np.testing.assert_array_equal(z, y[:part])
