"""The MLP loss and gradient at the edges of its 64-sample tiles and past the 512 partials of one round
(32768 samples), against the FP64 oracle.

Tolerance: an FP32 chain of the longest product (64 terms), its bias and the feature sum (8) is off by
at most (64 + 64 + 8) 2^-24 = 8e-6 of its terms; a gradient has two such chains in it (forward pass and
delta), 1.6e-5, and its sum over the samples adds 64 2^-24 = 4e-6: 2e-5 of the largest entry.  The
targets are kept off the predictions, so that no residual is a small difference."""
import numpy as np
import pytest

import librpa_amd as L
from oracle import mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 130, 32768, 32769, 70001])
def test_tile_edges(lib, n):
    print(f"mlp loss and gradient, n = {n}", flush=True)
    rng = np.random.default_rng(n)
    p = (mlp.init_params(3) + 0.05 * rng.standard_normal(mlp.NPARAM)).astype(np.float32)
    X = rng.standard_normal((n, mlp.NFEAT)).astype(np.float32)
    t = (5.0 + rng.uniform(0.0, 1.0, n)).astype(np.float32)
    loss, g = L.mlp_loss_grad(p, X, t)
    loss64, g64 = mlp.loss_and_grad(p.astype(np.float64), X.astype(np.float64), t.astype(np.float64))
    print(f"  loss {loss:.8f} / {loss64:.8f}, max |dg| {np.abs(g - g64).max():.2e} of {np.abs(g64).max():.2e}")
    assert abs(loss - loss64) <= 2e-5 * loss64
    assert np.abs(g - g64).max() <= 2e-5 * np.abs(g64).max()
