"""Householder QR through ttf_dqr at the shapes where its panels can go
wrong: one column and one row, panels of 31 to 33 columns, rows around the
register slabs (64, 256, 512, 768, 1024) and past them, wide matrices, zero
columns and rank-deficient ones.

Backward stability: |Q R - A| and |Q^T Q - I| are within a small multiple of
the column count times eps (64 columns, factor 10); the signs are LAPACK's,
so Q and R match numpy's where the matrix has full rank and modest condition.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _qr(A):
    import ttfort
    lib = ttfort.load()
    n, m = A.shape
    k = min(n, m)
    d = ttfort.DeviceArray.from_numpy(A)
    R = ttfort.DeviceArray((k, m))
    ttfort.check(lib.ttf_dqr(n, m, d.ptr, R.ptr, k), lib)
    return d.numpy().reshape(-1, order="F")[:n * k].reshape((n, k), order="F"), R.numpy()


@pytest.mark.parametrize("n,m", [(1, 1), (5, 1), (1, 7), (31, 31), (40, 32), (64, 33), (65, 20), (256, 64), (257, 63),
                                 (512, 96), (513, 40), (768, 32), (769, 5), (1024, 70), (1025, 40), (48, 100)])
def test_qr_shapes(ttlib, n, m):
    rng = np.random.default_rng(n + m)
    A = rng.standard_normal((n, m))
    Q, R = _qr(A)
    k, eps = min(n, m), np.finfo(float).eps
    tol = 10 * max(k, 8) * eps
    assert np.abs(Q.T @ Q - np.eye(k)).max() <= tol
    assert np.linalg.norm(Q @ R - A) <= tol * np.linalg.norm(A)
    assert np.array_equal(R, np.triu(R))
    Rn = np.linalg.qr(A)[1]
    assert np.linalg.norm(R - Rn) <= 1e-10 * np.linalg.norm(Rn)


def test_qr_rank_deficient(ttlib):
    rng = np.random.default_rng(3)
    A = rng.standard_normal((300, 9)) @ rng.standard_normal((9, 50))
    A[:, 4] = 0.0
    A[:, 40] = A[:, 41]
    Q, R = _qr(A)
    tol = 500 * np.finfo(float).eps
    assert np.abs(Q.T @ Q - np.eye(50)).max() <= tol
    assert np.linalg.norm(Q @ R - A) <= tol * np.linalg.norm(A)
