"""The one-sided Jacobi's pair step from Gram matrices and the rotations of
small symmetric matrices, where their tiles and lanes end: odd column counts,
a last block that is short or empty, rows that are no multiple of a wave's
16, so many rows that a pair holds fewer columns than 32 or only two, columns
graded over 12 decades, and data far from one.

Bars: singular values to 5e-13 of the largest and the short side's vectors
orthonormal to 1e-12, those of the other truncation tests; eigenvalues and
residuals to 64 eps of the norm times the order, the rounding of a few sweeps
of n rotations a row.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,q", [(2, 2), (5, 3), (33, 17), (40, 31), (100, 33), (257, 63), (300, 256), (515, 65),
                                 (600, 513), (3000, 9)])
@pytest.mark.parametrize("grade,scale", [(0.0, 1.0), (12.0, 1.0), (3.0, 1e120), (3.0, 1e-120)])
def test_pairs(ttlib, p, q, grade, scale):
    import ttfort
    rng = np.random.default_rng(1000 * p + q)
    A = rng.standard_normal((p, q)) * 10.0 ** -rng.uniform(0.0, grade, q) * scale
    s, O, kpos, _ = ttfort.svd_side(A, "R")
    sr = np.linalg.svd(A, compute_uv=False)
    assert np.abs(s - sr).max() <= 5e-13 * sr[0]
    V = O[:, :kpos] if O.shape[0] == q else O[:kpos].T
    assert np.abs(V.T @ V - np.eye(kpos)).max() <= 1e-12


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 25, 26, 27, 28, 31, 32, 33, 47, 63, 64])
def test_orders(ttlib, n):
    import ttfort
    rng = np.random.default_rng(n)
    A = rng.standard_normal((2, n, n))
    A = A + A.transpose(0, 2, 1)
    A[1] *= np.outer(10.0 ** -np.arange(n) , np.ones(n)) ** 0.1
    A[1] = A[1] + A[1].T
    w, Q = ttfort.syev_small(A.copy())
    for a, wi, qi in zip(A, w, Q):
        tol = 64 * n * np.finfo(float).eps
        assert np.abs(wi - np.linalg.eigvalsh(a)).max() <= tol * np.linalg.norm(a)
        assert np.abs(qi.T @ qi - np.eye(n)).max() <= tol
        assert np.abs(a @ qi - qi * wi).max() <= tol * np.linalg.norm(a)


@pytest.mark.parametrize("n", [60, 64])
def test_rotations_orthogonal(ttlib, n):
    """Ten sweeps give every column 10 (n - 1) rotations, each of which may
    miss c^2 + s^2 = 1 by its rounding, eps: at random signs
    ||Q^T Q - I||_F = sqrt(n * 10 (n - 1)) eps, over 32 matrices on average."""
    import ttfort
    rng = np.random.default_rng(n)
    A = rng.standard_normal((32, n, n))
    _, Q = ttfort.syev_small(A + A.transpose(0, 2, 1))
    miss = np.mean([np.linalg.norm(q.T @ q - np.eye(n)) for q in Q])
    assert miss <= np.sqrt(10.0 * n * (n - 1)) * np.finfo(float).eps


@pytest.mark.parametrize("n", [4, 27, 32, 33, 64])
@pytest.mark.parametrize("scale", [1e-153, 1e-156, 1e-158])
def test_rotations_of_tiny_entries(ttlib, n, scale):
    """Entries whose squares are subnormal: the rotations' angles lose digits
    with d^2 + 4 a^2, their orthogonality does not."""
    import ttfort
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    _, Q = ttfort.syev_small(((a + a.T) * scale)[None])
    assert np.abs(Q[0].T @ Q[0] - np.eye(n)).max() <= 64 * n * np.finfo(float).eps
