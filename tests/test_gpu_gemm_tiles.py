"""The GEMM engine's tile kernels at the sizes where they can go wrong: rows
and columns around every tile edge, K around its chunk and split lengths,
16-byte loads against operands that are not aligned for them, and a
bound-exact comparison with numpy.

The products run through the phi2 updates (tt_linalg.f90:315-340): the left
one multiplies two transposed operands (contiguous along K), the right one a
row-contiguous operand and a transposed one.  |computed - exact| is at most
K eps |A| |B| per product to first order; the two chained products and the
reference's own rounding are covered by 2 (K1 + K2 + 2) eps on the product of
absolute values.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1, 1, 1), (15, 17, 16, 1, 33), (64, 64, 64, 2, 64), (65, 63, 127, 1, 129), (128, 96, 40, 3, 97),
         (130, 31, 1000, 2, 66), (33, 200, 18, 5, 80), (2, 2, 514, 64, 2), (96, 128, 256, 1, 192),
         (192, 16, 30, 1, 16)]


def _run(side, dims, shift):
    import ttfort
    lib = ttfort.load()
    rx1, rx2, ry1, n, ry2 = dims
    rng = np.random.default_rng(sum(dims))
    if side == "left":
        p = rng.standard_normal((ry1, rx1))
        out_shape = (ry2, rx2)
    else:
        p = rng.standard_normal((rx2, ry2))
        out_shape = (rx1, ry1)
    x, y = rng.standard_normal((rx1, n, rx2)), rng.standard_normal((ry1, n, ry2))

    def dev(a):   # `shift` doubles into an allocation: 8 bytes off the 16-byte grid when odd
        d = ttfort.DeviceArray((a.size + shift,))
        d.upload(np.concatenate([np.zeros(shift), a.reshape(-1, order="F")]))
        return d

    d = [dev(a) for a in (p, x, y)]
    out = ttfort.DeviceArray(out_shape)
    fn = lib.ttf_dphi2_left if side == "left" else lib.ttf_dphi2_right
    ttfort.check(fn(rx1, rx2, ry1, n, ry2, *[ctypes.c_void_p(a.ptr + 8 * shift) for a in d], out.ptr), lib)

    def chain(p, x, y):
        if side == "left":
            return np.einsum("cbj,bja->ca", np.einsum("gb,gjc->cbj", p, y, optimize=True), x, optimize=True)
        return np.einsum("bjc,gjc->bg", np.einsum("bja,ac->bjc", x, p, optimize=True), y, optimize=True)

    k = (ry1 + rx1 * n) if side == "left" else (rx2 + n * ry2)
    bound = 2 * (k + 2) * np.finfo(float).eps * chain(abs(p), abs(x), abs(y))
    return out.numpy(), chain(p, x, y), bound


@pytest.mark.parametrize("side", ["left", "right"])
@pytest.mark.parametrize("dims", SIZES)
def test_gemm_tile_edges(ttlib, side, dims):
    aligned, ref, bound = _run(side, dims, 0)
    assert np.all(np.abs(aligned - ref) <= bound)
    shifted, _, _ = _run(side, dims, 1)
    assert np.array_equal(aligned, shifted)   # the same sums in the same order


def test_tuning_follows_the_load_mode(ttlib):
    """A tile timed on aligned operands is not taken over for operands that
    are read element by element, nor the other way round; each is tuned once."""
    dims = (200, 72, 136, 3, 104)   # sizes no other test uses
    tuned = []
    for shift in (0, 1, 0, 1):
        before = ttlib.ttf_autotune_count()
        _run("left", dims, shift)
        tuned.append(ttlib.ttf_autotune_count() - before)
    assert tuned[0] > 0 and tuned[1] > 0 and tuned[2:] == [0, 0]


# rx1, m, rx2, ry1, n, ry2, ra1, ra2; modes past 8 keep the three products
F32_SIZES = [(1, 1, 1, 1, 9, 1, 1, 1), (16, 1, 36, 33, 9, 20, 1, 1), (63, 1, 8, 64, 12, 5, 2, 2),
             (64, 1, 65, 65, 9, 13, 3, 1), (13, 5, 64, 66, 10, 3, 5, 4), (32, 2, 100, 130, 9, 7, 4, 3),
             (65, 2, 12, 31, 11, 9, 3, 2), (128, 1, 4, 128, 16, 6, 1, 5), (66, 3, 33, 96, 9, 11, 2, 7),
             (20, 1, 516, 17, 9, 2, 30, 9), (48, 4, 128, 192, 20, 4, 3, 3)]


@pytest.mark.parametrize("dims", F32_SIZES)
def test_gemm_tile_edges_f32(ttlib, dims):
    """The same edges in FP32, four elements to a load, through the three
    products of ttf_sbfun3: operands of which one can be read 16 bytes at a
    time and the other not, K around its chunk (32 and 64) and split lengths,
    and every operand one element off the 16-byte grid.  Per stage the error
    is at most (K + 2) eps of the sum of absolute values."""
    import ttfort
    rx1, m, rx2, ry1, n, ry2, ra1, ra2 = dims
    assert ttfort.bfun3_route(dims, 1, np.float32) == "chain"
    rng = np.random.default_rng(sum(dims))
    ops = [rng.standard_normal(s).astype(np.float32)
           for s in ((ry1, rx1, ra1), (ra1, n, m, ra2), (rx2, ra2, ry2), (rx1, m, rx2))]

    def product(shift):
        dev = []
        for a in ops:
            dev.append(ttfort.DeviceArray((a.size + shift,), np.float32))
            dev[-1].upload(np.concatenate([np.zeros(shift, np.float32), a.reshape(-1, order="F")]))
        out = ttfort.DeviceArray((ry1 * n * ry2 + shift,), np.float32)
        p = [ctypes.c_void_p(a.ptr + 4 * shift) for a in dev + [out]]
        ttfort.check(ttlib.ttf_sbfun3(*dims, 1, *p[:4], rx1 * m * rx2, p[4], ry1 * n * ry2), ttlib)
        return out.numpy()[shift:].reshape((ry1, n, ry2), order="F")

    def chain(p1, A, p2, x):
        t = np.einsum("bjd,dac->bjac", x, p2, optimize=True)
        t = np.einsum("fija,bjac->bfic", A, t, optimize=True)
        return np.einsum("gbf,bfic->gic", p1, t, optimize=True)

    got = product(0)
    wide = [a.astype(np.float64) for a in ops]
    bound = (rx2 + m * ra2 + rx1 * ra1 + 6) * np.finfo(np.float32).eps * chain(*[abs(a) for a in wide])
    assert np.all(np.abs(got - chain(*wide)) <= bound)
    assert np.array_equal(got, product(1))   # the same sums in the same order
