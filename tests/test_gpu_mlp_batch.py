"""Loss and gradient of the learned preconditioner at the batch sizes where
its kernels can go wrong: one column, tile edges of 32 columns, gradient
slices of 128 columns and the largest number of slices, and features that
are not on a 16-byte boundary.

Against the oracle in 64 bits: every sum has at most K = 4096 + 256 terms of
fp32 rounding 2^-24, accumulated in chunks, so the 2-norm of the gradient is
held to 1e-5 and the loss (summed in 64 bits from fp32 outputs) to 1e-6.
"""
import ctypes

import numpy as np
import pytest

from oracle import mlp as ML

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 31, 33, 64, 129, 2047, 4100])
def test_loss_grad_batch_sizes(ttlib, M):
    import ttfort
    rng = np.random.default_rng(M)
    theta = rng.uniform(-0.08, 0.08, ML.n_params()).astype(np.float32)
    ttfort.mlp_set_params(theta)
    X = rng.standard_normal((256, M)).astype(np.float32)
    X[:64] = 1.0 + 0.2 * rng.uniform(-1.0, 1.0, (64, M))   # block diagonals, which the skip term divides by
    T = rng.standard_normal((64, M)).astype(np.float32)
    loss, g = ttfort.mlp_loss_grad(X, T)
    y, cache = ML.forward(theta, X, round_weights=True, dtype=np.float64)
    ref = ML.backward(cache, y, T)
    assert abs(loss - ML.loss(y, T)) <= 1e-6 * ML.loss(y, T)
    assert np.linalg.norm(g - ref) <= 1e-5 * np.linalg.norm(ref)
    # features 4 bytes past a 16-byte boundary
    dX, dT = ttfort.DeviceArray((X.size + 1,), np.float32), ttfort.DeviceArray.from_numpy(T.reshape(-1, order="F"))
    dX.upload(np.concatenate([np.zeros(1, np.float32), X.reshape(-1, order="F")]))
    loss2, g2 = ctypes.c_double(), np.empty_like(g)
    ttfort.check(ttlib.ttf_mlp_loss_grad(M, ctypes.c_void_p(dX.ptr + 4), dT.ptr, ctypes.byref(loss2), g2.ctypes.data),
                 ttlib)
    assert loss2.value == loss and np.array_equal(g, g2)
