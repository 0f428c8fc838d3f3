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
