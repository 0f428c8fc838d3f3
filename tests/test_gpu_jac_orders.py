"""Block-Jacobi 'c' blocks at the orders where the register tiles of the
symmetric inverse change (16 TS = 32, 64, 128) and one past them, for
operators whose blocks are positive definite, and for non-symmetric ones
that take the pivoting inverse, with one and with many bond pairs.

Against the oracle (LU-based): condition numbers are below 20, so 1e-10
relative covers the rounding of both inverses at order 128.
"""
import numpy as np
import pytest

from oracle import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("rx1,n,rx2,ra1,ra2", [(1, 1, 1, 1, 1), (3, 2, 5, 1, 2), (5, 31, 4, 3, 3), (2, 32, 3, 2, 2),
                                               (3, 33, 2, 6, 6), (4, 64, 5, 6, 6), (2, 65, 2, 2, 3), (1, 127, 3, 2, 1),
                                               (2, 128, 1, 2, 2), (40, 3, 33, 2, 2)])
def test_djac_c_orders(ttlib, rx1, n, rx2, ra1, ra2, symmetric):
    import ttfort
    rng = np.random.default_rng(n)
    P1 = 0.2 * rng.standard_normal((rx1, rx1, ra1))
    P2 = 0.2 * rng.standard_normal((rx2, ra2, rx2))
    P1[:, :, 0] = np.eye(rx1)
    P2[:, 0, :] = np.eye(rx2)
    A = rng.standard_normal((ra1, n, n, ra2)) / (4.0 * np.sqrt(n * ra1 * ra2))
    if symmetric:
        A = 0.5 * (A + np.transpose(A, (0, 2, 1, 3)))
    A[0, :, :, 0] += 2.0 * np.eye(n)
    phi1, Af, phi2 = K._flat(P1), K._flat(A), K._flat(P2)
    J = ttfort.djac_gen("c", rx1, n, rx2, ra1, ra2, phi1, Af, phi2)
    Jr = K.djac_gen("c", rx1, n, rx2, ra1, ra2, phi1, Af, phi2)
    assert np.abs(J - Jr).max() <= 1e-10 * np.abs(Jr).max()
