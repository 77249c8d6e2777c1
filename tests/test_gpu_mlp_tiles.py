"""The training kernel at the edges of its sample tiles (32) and of its grid (256 workgroups of a
tile each: 8192 samples), every block of the gradient against the FP64 numpy oracle.

Tolerance: a hidden unit is a dot product of at most 65 FP32 terms and a tanh, so about 66
roundings of 2^-24 = 4e-6; the gradient passes two such layers and one back: 1.2e-5 of a block's
norm, where the block's terms do not cancel; 1e-4 leaves room for cancelling ones."""
import numpy as np
import pytest

from gplum_amd import gpu
from oracle import mlp as omlp

pytestmark = pytest.mark.gpu

BLOCKS = {"W1": (0, 256), "b1": (256, 320), "W2": (320, 4416), "b2": (4416, 4480), "w3": (4480, 4544), "b3": (4544, 4545)}


@pytest.mark.parametrize("n", [2, 31, 32, 33, 8191, 8192, 8193, 16385])
def test_gradient_blocks_at_tile_edges(n):
    rng = np.random.default_rng(n)
    x = rng.normal(0.0, 1.0, (n, 4)).astype(np.float32).astype(np.float64)
    y = rng.poisson(np.exp(1.0 + 0.7 * x[:, 0])).astype(np.float64)
    theta = omlp.init_params(seed=4).astype(np.float32).astype(np.float64)
    loss, grad = gpu.mlp_loss_grad(theta, x, y)
    loss_o, grad_o = omlp.loss_and_grad(theta, x, y)
    assert abs(loss - loss_o) <= 1e-6 * abs(loss_o) + 1e-9
    for name, (a, b) in BLOCKS.items():
        err = np.linalg.norm(grad[a:b] - grad_o[a:b]) / np.linalg.norm(grad_o[a:b])
        print("n %d %s gradient error %.2e" % (n, name, err))
        assert err < 1e-4
