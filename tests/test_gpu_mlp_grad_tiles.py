"""The training gradient on the matrix cores at the edges of its 16-sample
tiles and of its one-block-per-CU grid (4,096 samples fill it once; beyond, a
block accumulates several tiles), against the FP64 oracle.  A gradient entry is
a sum of n products of FP32 numbers through four layers: its FP32 error grows
as the square root of the terms, far below 1e-5 of the norm at these sizes."""
import numpy as np
import pytest

from oracle import farfield as FF
from pawan_amd import capi, workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 4095, 4096, 4097, 9000])
def test_gradient(n):
    rng = np.random.default_rng(n)
    params = np.zeros(capi.MLP_PARAMS, dtype=np.float32)
    for name, (o, size) in FF.OFF.items():
        fan_in = 16 if name == "W1" else 128
        params[o:o + size] = rng.normal(size=size) * (0.8 / np.sqrt(fan_in) if name[0] == "W" else 0.1)
    X = rng.normal(size=(n, 16)).astype(np.float32)
    Y = rng.normal(size=(n, 12)).astype(np.float32)
    with capi.Solver(W.ring_1k()) as g:
        g.ff_set_weights(params)
        grad, loss = g.ff_mlp_grad(X, Y)
        again, loss2 = g.ff_mlp_grad(X, Y)  # the kept buffers
    np.testing.assert_array_equal(grad, again)
    assert loss == loss2
    lo, go = FF.mlp_loss_grad(params.astype(np.float64), X.astype(np.float64), Y.astype(np.float64))
    assert loss == pytest.approx(lo, rel=1e-5)
    for name, (o, size) in FF.OFF.items():
        a, b = grad[o:o + size], go[o:o + size]
        assert np.linalg.norm(a - b) < 1e-5 * np.linalg.norm(b), name
