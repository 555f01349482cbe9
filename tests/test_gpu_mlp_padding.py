"""The lanes past the last sample of the MLP gradient's 64-sample tile hold x = 0: with parameters whose
hidden units overflow there, and for no sample, the gradient stays that of the samples.

Tolerance: with one feature in use and all units alike the sums have at most 64 equal terms, 64 x 2^-24 =
4e-6 of each value."""
import numpy as np
import pytest

import librpa_amd as L
from oracle import mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 65])
def test_padding_lanes(lib, n):
    print(f"mlp padding lanes, n = {n}", flush=True)
    p = np.zeros(mlp.NPARAM, dtype=np.float32)
    w1, b1, w2 = p[:512].reshape(8, 64), p[512:576], p[576:576 + 4096]
    b2, w3 = p[4672:4736], p[4736:4800]
    w1[0], b1[:], w2[:], b2[:], w3[:] = 1e20, 1e20, 1e20, 0.3, 0.1
    X = np.zeros((n, mlp.NFEAT), dtype=np.float32)
    X[:, 0] = -1.0  # z1 = 0 for every sample, 1e20 at x = 0
    t = np.full(n, 5.0, dtype=np.float32)
    loss, g = L.mlp_loss_grad(p, X, t)
    loss64, g64 = mlp.loss_and_grad(p.astype(np.float64), X.astype(np.float64), t.astype(np.float64))
    assert abs(loss - loss64) <= 4e-6 * loss64
    assert np.all(np.isfinite(g))
    assert np.all(np.abs(g - g64) <= 4e-6 * np.abs(g64))
