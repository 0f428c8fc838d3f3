"""The route that a local matvec takes (ttf_bfun3_route), which is decided on
the host: each kernel's own shapes, the switches that take a kernel out, and
the refusals of the call.  Runs without a GPU."""
import os
import subprocess
import sys

import numpy as np
import pytest

import ttfort

TYPES = [np.float64, np.float32, np.complex128, np.complex64]
BLOCK = (128, 2, 128, 128, 2, 128, 5, 5)     # a spin chain's largest local problem
WIDE = (64, 64, 64, 64, 64, 64, 6, 6)        # modes past the one-launch kernels


@pytest.mark.parametrize("dtype", TYPES)
def test_routes(dtype):
    assert ttfort.bfun3_route((2, 2, 4, 2, 2, 4, 5, 5), 1, dtype) == "small"
    assert ttfort.bfun3_route(BLOCK, 1, dtype) == "small"
    assert ttfort.bfun3_route(BLOCK, 16, dtype) == ("fused" if dtype is np.float64 else "chain")
    assert ttfort.bfun3_route(WIDE, 1, dtype) == "chain"


def test_switches():
    code = ("import numpy as np, ttfort\n"
            "print(ttfort.bfun3_route(%r, 1), ttfort.bfun3_route(%r, 1, np.float32))" % (BLOCK, BLOCK))
    env = dict(os.environ, PYTHONPATH=os.path.dirname(ttfort.__file__), TTF_BFUN3_SMALL="0")
    for fused, want in (("1", "fused chain"), ("0", "chain chain")):
        r = subprocess.run([sys.executable, "-c", code], env=dict(env, TTF_BFUN3_FUSED=fused), capture_output=True,
                           text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-2000:]
        assert r.stdout.strip() == want


def test_refusals():
    lib = ttfort.load()
    route = ttfort.C.c_int(7)
    for kind, sizes, nvec, out in ((b"q", BLOCK, 1, route), (b"d", (0,) + BLOCK[1:], 1, route), (b"d", BLOCK, 0, route),
                                   (b"d", BLOCK, 1, None)):
        assert lib.ttf_bfun3_route(kind, *sizes, nvec, ttfort.C.byref(out) if out is not None else None) != 0
        lib.ttf_clear_error()
    assert route.value == 7


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("left,n,right,ra,nvec", [(512, 2, 2, 3, 1), (512, 2, 1, 3, 1), (384, 2, 4, 5, 1), (400, 2, 8, 3, 1)])
def test_few_large_groups_spread(dtype, left, n, right, ra, nvec):
    """A long left rank and a short right one would leave the one-launch
    kernel a work-group or a few, each with the whole of Phi1 to read: the
    product spreads over the chip the other way."""
    shape = (left, n, right, left, n, right, ra, ra)
    assert ttfort.bfun3_route(shape, nvec, dtype) != "small"


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("left,n,right,ra,nvec", [(2, 2, 400, 5, 1), (4, 2, 400, 3, 1), (64, 2, 1, 5, 1), (64, 2, 64, 5, 1),
                                                  (128, 2, 4, 5, 1), (32, 2, 32, 5, 8)])
def test_many_or_small_groups_stay(dtype, left, n, right, ra, nvec):
    shape = (left, n, right, left, n, right, ra, ra)
    assert ttfort.bfun3_route(shape, nvec, dtype) == "small"


@pytest.mark.parametrize("dtype", TYPES)
def test_more_groups_than_a_batch(dtype):
    """The chains take at most 65535 products in a batch."""
    assert ttfort.bfun3_route((1, 2, 1, 1, 2, 70000, 2, 2), 1, dtype) == "small"
