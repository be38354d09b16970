"""Edges of the cache kernels' tiles against the CPU oracle: inference tiles of 256 samples
(64 per wave, 16 per matrix tile) looped over by 768 blocks, training tiles of 64 samples
(16 per wave) looped over by 256 blocks, each of which writes one gradient partial.

Tolerances are those of test_gpu_nrc.py: features, weights and activations are rounded to
bf16 on both sides and a rounding may flip where FP32 and FP64 sums straddle a boundary.
"""
import numpy as np
import pytest

import nrc_oracle as N
from crender_amd import Context, Nrc
from test_gpu_nrc import _queries

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nrc():
    ctx = Context(0)
    m = Nrc(ctx, max_batch=32_768, seed=5)
    yield m
    m.close()
    ctx.close()


@pytest.mark.parametrize("n", [15, 17, 255, 257, 768 * 256 + 1])
def test_forward_tiles(nrc, n):
    q = _queries(n, n)
    got = nrc.infer(q)
    ref = N.forward(nrc.params(), N.encode(q, True), True)[0][:, :3]
    assert np.isclose(got, ref, rtol=1e-2, atol=1e-3).mean() >= 0.995
    assert np.abs(got - ref).max() < 5e-2 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("n", [16, 63, 65, 129, 256 * 64 + 65])
def test_gradient_tiles(nrc, n):
    q = _queries(n, n + 1)
    t = (np.random.default_rng(n).random((n, 3)) * 2).astype(np.float32)
    loss, g = nrc.gradient(q, t)
    lref, gref = N.loss_and_grad(nrc.params(), q, t, round_bf16=True)
    assert abs(loss - lref) <= 2e-2 * abs(lref)
    for o, (k, c) in zip(N.offsets(), N.LAYERS):
        a, b = g[o:o + k * c].astype(np.float64), gref[o:o + k * c]
        assert np.linalg.norm(a - b) < 3e-2 * max(np.linalg.norm(b), 1e-30), (o, n)
