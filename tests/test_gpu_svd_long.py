"""Long-side singular vectors (Cholesky QR of T V / s) at the orders where the
register tiles of the Cholesky inverse change: 32, 64, 128 and their
neighbours, and one past the Cholesky path.

Columns of modest condition: orthonormal to 1e-12, the residual of A V to
1e-12 of the largest singular value and singular values to 5e-13 of it, the
bars of the other truncation tests.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q", [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129])
@pytest.mark.parametrize("wide", [False, True])
def test_long_side_vectors(ttlib, q, wide):
    import ttfort
    rng = np.random.default_rng(q)
    A = rng.standard_normal((q + 170, q)) * 10.0 ** rng.uniform(-1.0, 0.0, q)
    s, O, kpos, _ = ttfort.svd_side(A.T if wide else A, "R" if wide else "L")
    sr = np.linalg.svd(A, compute_uv=False)
    assert kpos == q and np.abs(s - sr).max() <= 5e-13 * sr[0]
    assert np.abs(O.T @ O - np.eye(q)).max() <= 1e-12
    # A^T O has orthogonal columns of lengths s
    W = A.T @ O
    assert np.abs(W.T @ W - np.diag(sr ** 2)).max() <= 1e-12 * sr[0] ** 2
