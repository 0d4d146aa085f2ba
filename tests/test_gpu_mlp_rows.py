"""Training kernels at the batch sizes where their row groups end: fewer rows
than the forward pass's 16-row tile or the backward pass's 64-row group,
remainders of both, as many groups as the gradient reduction loads at once (128)
and more.

Bound: every FP32 sum of terms t is within (terms in its chain + 100) 2^-24
sum|t| of the FP64 oracle's, the 100 covering the terms' own rounding (the
64-term inner products and GELU's exponential, a few ulp each).
"""
import numpy as np
import pytest

from gpuimogen_amd import abi, learned_drag as L
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 15, 16, 17, 63, 64, 65, 2048, 8192, 8193, 20000])
def test_rows(batch):
    rng = np.random.default_rng(batch)
    p = L.init_params(rng)
    p[mo.OFF_B1:mo.OFF_W2] = rng.normal(0, 0.1, 64)
    p[mo.OFF_B2:mo.OFF_W3] = rng.normal(0, 0.1, 64)
    x = rng.normal(0, 1, (batch, 5)).astype(np.float32)
    dy = rng.normal(0, 1, (batch, 3)).astype(np.float32)
    P, X, DY = (L.DeviceArray.from_host(a) for a in (p, x, dy))
    act, y = L.DeviceArray((batch, 256), np.float32), L.DeviceArray((batch, 3), np.float32)
    g = L.DeviceArray((mo.NPARAMS,), np.float32)
    print(f"batch {batch}", flush=True)
    abi.call("imogen_mlp_forward", P.ptr(), batch, X.ptr(), act.ptr(), y.ptr())
    abi.call("imogen_mlp_backward", P.ptr(), batch, X.ptr(), act.ptr(), DY.ptr(), g.ptr())
    p64, x64, d64 = p.astype(np.float64), x.astype(np.float64), dy.astype(np.float64)
    yr, cache = mo.forward(p64, x64)
    eps = 2.0 ** -24
    W1, b1, W2, b2, W3, b3 = mo.unpack(p64)
    z1, h1, z2, h2 = cache
    assert np.all(np.abs(y.to_host() - yr) <= 164 * eps * (np.abs(h2) @ np.abs(W3) + np.abs(b3) + 1))
    for k, ref in enumerate(cache):
        assert np.abs(act.to_host()[:, 64 * k:64 * (k + 1)] - ref).max() <= 164 * eps * (1 + np.abs(ref).max() * 8)
    ref = mo.backward(p64, x64, cache, d64)
    a2 = (np.abs(d64) @ np.abs(W3).T) * (np.abs(mo.gelu_grad(z2)) + 1)
    a1 = (a2 @ np.abs(W2).T) * (np.abs(mo.gelu_grad(z1)) + 1)
    mag = np.zeros(mo.NPARAMS)
    mag[mo.OFF_W1:mo.OFF_B1] = (np.abs(x64).T @ a1).ravel()
    mag[mo.OFF_B1:mo.OFF_W2] = a1.sum(0)
    mag[mo.OFF_W2:mo.OFF_B2] = ((np.abs(h1) + 1).T @ a2).ravel()
    mag[mo.OFF_B2:mo.OFF_W3] = a2.sum(0)
    mag[mo.OFF_W3:mo.OFF_B3] = ((np.abs(h2) + 1).T @ np.abs(d64)).ravel()
    mag[mo.OFF_B3:] = np.abs(d64).sum(0)
    chain = 64 + -(-batch // 64)
    err = np.abs(g.to_host() - ref)
    print("worst share of the bound", (err / ((chain + 100) * eps * mag)).max(), flush=True)
    assert np.all(err <= (chain + 100) * eps * mag)
