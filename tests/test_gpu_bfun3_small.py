"""The one-launch local matvec on the vector units: every column bucket of
its narrow operands (2, 3, 5, 8), row counts around the wave and work-group
sizes (63, 64, 65, 511, 513 rows and more), rectangular operators, several
vectors with padded leading dimensions, and an output that overlaps the
input, which the general path takes.

Against numpy in 64 bits: a sum of K terms, in parts and then over the
parts, is within (K + 4) eps of the sum of absolute values per stage (twice
that for complex products).
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FN = {np.float64: "ttf_dbfun3", np.float32: "ttf_sbfun3", np.complex128: "ttf_zbfun3", np.complex64: "ttf_cbfun3"}
# rx1, m, rx2, ry1, n, ry2, ra1, ra2, nvec
SHAPES = [(1, 1, 1, 1, 1, 1, 1, 1, 1), (2, 2, 4, 2, 2, 4, 5, 5, 1), (21, 3, 7, 21, 3, 7, 3, 3, 2),
          (32, 2, 9, 5, 4, 6, 4, 2, 1), (13, 5, 3, 65, 8, 2, 8, 7, 1), (73, 7, 17, 33, 2, 3, 2, 8, 3),
          (57, 9, 5, 513, 5, 2, 1, 5, 1), (64, 2, 64, 64, 2, 3, 3, 3, 1), (3, 8, 130, 200, 6, 1, 6, 6, 1)]


def _chain(shape, p1, A, p2, x):
    t = np.einsum("bjdv,dac->bjacv", x, p2, optimize=True)
    t = np.einsum("fija,bjacv->bficv", A, t, optimize=True)
    return np.einsum("gbf,bficv->gicv", p1, t, optimize=True)


@pytest.mark.parametrize("dtype", list(FN))
@pytest.mark.parametrize("dims", SHAPES)
def test_small_matvec(ttlib, dims, dtype):
    import ttfort
    rx1, m, rx2, ry1, n, ry2, ra1, ra2, nvec = dims
    rng = np.random.default_rng(sum(dims))

    def draw(*s):
        a = rng.standard_normal(s)
        return (a + 1j * rng.standard_normal(s) if np.dtype(dtype).kind == "c" else a).astype(dtype)

    p1, A, p2 = draw(ry1, rx1, ra1), draw(ra1, n, m, ra2), draw(rx2, ra2, ry2)
    nx, ny, pad = rx1 * m * rx2, ry1 * n * ry2, 3 if nvec > 1 else 0
    x = draw(rx1, m, rx2, nvec)
    xs = np.zeros((nx + pad, nvec), dtype)
    xs[:nx] = x.reshape(nx, nvec, order="F")
    dev = [ttfort.DeviceArray.from_numpy(a.reshape(-1, order="F")) for a in (p1, A, p2, xs)]
    dy = ttfort.DeviceArray((ny + pad, nvec), dtype)
    dy.upload(np.full((ny + pad, nvec), 7, dtype))
    fn = getattr(ttlib, FN[dtype])
    ttfort.check(fn(*dims[:8], nvec, *[d.ptr for d in dev], nx + pad, dy.ptr, ny + pad), ttlib)
    y = dy.numpy()
    wide = [a.astype(np.complex128 if a.dtype.kind == "c" else np.float64) for a in (p1, A, p2, x)]
    ref = _chain(dims, *wide).reshape(ny, nvec, order="F")
    bound = _chain(dims, *[abs(a) for a in wide]).reshape(ny, nvec, order="F")
    k = rx2 + m * ra2 + rx1 * ra1 + 12
    assert np.all(np.abs(y[:ny] - ref) <= 2 * k * np.finfo(dtype).eps * bound)
    assert np.all(y[ny:] == 7)          # nothing past the columns


def test_overlapping_output(ttlib):
    """y = B x in place (one vector, leading dimensions not used and given
    as 0): the general path stages the product."""
    import ttfort
    r, n, ra = 24, 2, 3
    rng = np.random.default_rng(1)
    p1, A, p2, x = (rng.standard_normal(s) + 1j * rng.standard_normal(s)
                    for s in ((r, r, ra), (ra, n, n, ra), (r, ra, r), (r, n, r)))
    dev = [ttfort.DeviceArray.from_numpy(a.reshape(-1, order="F")) for a in (p1, A, p2, x)]
    out = ttfort.DeviceArray((r * n * r,), np.complex128)
    for y in (out, dev[3]):
        ttfort.check(ttlib.ttf_zbfun3(r, n, r, r, n, r, ra, ra, 1, *[d.ptr for d in dev], 0,
                                      ctypes.c_void_p(y.ptr), 0), ttlib)
    assert np.allclose(dev[3].numpy(), out.numpy(), rtol=1e-12, atol=1e-12 * np.abs(out.numpy()).max())
