"""The one-launch inference of the learned preconditioner at the sizes where
it can go wrong: fewer columns than a work-group's 16, one past it, blocks
that straddle right-interface indices, and more bond pairs (72) than the 64
coefficients staged at a time.

Against the oracle with the same roundings (bf16 weights and layer inputs):
an activation whose bf16 rounding flips on the fp32 summation order moves an
output by one bf16 step of one term, so 2e-3 of the largest output bounds
the difference, as in the forward-pass test.
"""
import numpy as np
import pytest

from oracle import mlp as ML

pytestmark = pytest.mark.gpu


def _theta(rng):
    return rng.uniform(-0.1, 0.1, ML.n_params()).astype(np.float32)


@pytest.mark.parametrize("M", [1, 15, 16, 17, 40])
def test_forward_columns(ttlib, M):
    import ttfort
    rng = np.random.default_rng(M)
    theta = _theta(rng)
    ttfort.mlp_set_params(theta)
    X = rng.standard_normal((256, M)).astype(np.float32)
    X[0, 0] = 0.0                        # no point-Jacobi term where the diagonal feature is zero
    Y = ttfort.mlp_forward(X)
    Yr, _ = ML.forward(theta, X, round_weights=True, dtype=np.float64, round_acts=True)
    assert np.abs(Y - Yr).max() <= 2e-3 * np.abs(Yr).max()


@pytest.mark.parametrize("rx1,rx2,ra1,ra2", [(1, 1, 1, 1), (3, 5, 2, 3), (17, 2, 9, 8), (16, 3, 1, 4), (7, 9, 6, 6)])
def test_precond_blocks(ttlib, rx1, rx2, ra1, ra2):
    import ttfort
    n, rng = 64, np.random.default_rng(rx1 + 100 * rx2)
    theta = _theta(rng)
    ttfort.mlp_set_params(theta)
    phi1 = rng.standard_normal(rx1 * rx1 * ra1)
    A = rng.standard_normal((ra1, n, n, ra2))
    A[0, :, :, 0] += 8.0 * np.eye(n)
    phi2 = rng.standard_normal(rx2 * ra2 * rx2)
    v = rng.standard_normal(rx1 * n * rx2)
    if rx1 > 2:
        v.reshape((rx1, n, rx2), order="F")[1, :, 0] = 0.0   # a zero residual slice
    args = (rx1, n, rx2, ra1, ra2, phi1, A.reshape(-1, order="F"), phi2, v)
    z = ttfort.mlp_precond(*args)
    X, sc = ML.features(*args)
    y, _ = ML.forward(theta, X.astype(np.float32), round_weights=True, dtype=np.float64, round_acts=True)
    ref = np.transpose((y * sc).reshape(n, rx1, rx2, order="F"), (1, 0, 2)).reshape(-1, order="F")
    assert np.abs(z - ref).max() <= 2e-3 * np.abs(ref).max()
