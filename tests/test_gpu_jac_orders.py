"""Block-Jacobi 'c' blocks at the orders where the register tiles of the
symmetric inverse change (16 TS = 32, 64, 128) and one past them, for
operators whose blocks are positive definite, and for non-symmetric ones
that take the pivoting inverse, with one and with many bond pairs, more left
indices than one slice of the blocks' intermediate holds, and an operator
rank past one batch of products.

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
                                               (2, 128, 1, 2, 2), (40, 3, 33, 2, 2), (130, 64, 1, 1, 20), (2, 1, 3, 1, 70000)])
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


def test_djac_c_scratch(ttlib):
    """Many blocks and large operator ranks: the scratch stays below the 64 MB
    of the intermediate (80 MB with the arena's headroom) and a few MB more,
    where bond pairs times blocks would be 1.15 GB."""
    import ctypes
    import ttfort
    hip = ctypes.CDLL("libamdhip64.so.7")

    def free():
        left, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(left), ctypes.byref(total)) == 0
        return left.value

    rx, n, ra = 300, 2, 40
    rng = np.random.default_rng(4)
    P1 = 0.01 * rng.standard_normal((rx, rx, ra))
    P2 = 0.01 * rng.standard_normal((rx, ra, rx))
    P1[:, :, 0] = np.eye(rx)
    P2[:, 0, :] = np.eye(rx)
    A = rng.standard_normal((ra, n, n, ra))
    A[0, :, :, 0] += 4.0 * np.eye(n)
    d = [ttfort.DeviceArray.from_numpy(K._flat(a)) for a in (P1, A, P2)]
    J = ttfort.DeviceArray((n * n * rx * rx,))
    ttfort.sync(ttlib)
    before = free()
    ttfort.check(ttlib.ttf_djac_gen(b"c", rx, n, rx, ra, ra, *[a.ptr for a in d], J.ptr), ttlib)
    ttfort.sync(ttlib)
    assert before - free() <= 96 << 20
    d1, d2 = np.einsum("bba->ba", P1), np.einsum("bab->ba", P2)
    M = np.einsum("ba,aijq,cq->bcij", d1, A, d2, optimize=True)
    got = J.numpy().reshape((n, n, rx, rx), order="F").transpose(3, 2, 0, 1)
    ref = np.linalg.inv(M)
    # 2 x 2 inverses: eps times the condition number, sums of 1600 terms
    tol = 1600 * np.finfo(float).eps * np.linalg.cond(M)[..., None, None] * np.abs(ref).max((2, 3), keepdims=True)
    assert np.all(np.abs(got - ref) <= tol)


def test_djac_c_range(ttlib):
    """Interfaces whose product alone would overflow: the sums over the left
    bond come first, as in the reference."""
    import ttfort
    rx1, n, rx2, ra = 3, 5, 4, 3
    rng = np.random.default_rng(5)
    P1, P2 = rng.uniform(0.5, 1.0, (rx1, rx1, ra)), rng.uniform(0.5, 1.0, (rx2, ra, rx2))
    A = 0.01 * rng.standard_normal((ra, n, n, ra)) + 2.0 * np.eye(n)[None, :, :, None]
    J = ttfort.djac_gen("c", rx1, n, rx2, ra, ra, K._flat(P1) * 2.0 ** 600, K._flat(A) * 2.0 ** -900,
                        K._flat(P2) * 2.0 ** 600)
    ref = K.djac_gen("c", rx1, n, rx2, ra, ra, K._flat(P1), K._flat(A), K._flat(P2)) * 2.0 ** -300
    assert np.abs(J - ref).max() <= 1e-12 * np.abs(ref).max()
