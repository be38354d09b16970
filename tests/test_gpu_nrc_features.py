"""The cache's input features, read through the network itself, and predictions far outside the
unit box.

With weights of 0 and +-1 the network passes three features through unchanged: the first layer
takes f into relu(f) and relu(-f), the hidden layers copy both, the output layer subtracts
them.  Every product is exact and every sum has one nonzero term, so the output is the bf16
feature itself.  The features are FP32 sines and cosines rounded to bf16: with an FP32 error of
at most 2 units in the last place (2^-22 relative) the result lies between the roundings of
the exact value moved by that much either way.
"""
import numpy as np
import pytest

import nrc_oracle as N
from crender_amd import Context, Nrc

pytestmark = pytest.mark.gpu

POSITIONS = {
    "unit": lambda g, n: g.random((n, 3)),
    # multiples of 2^-11: every argument is near a multiple of pi / 2
    "crossings": lambda g, n: g.integers(0, 2049, (n, 3)) / 2048.0,
    # on both sides of 16, beyond which the argument's reduction takes another way
    "edge": lambda g, n: 16.0 + g.uniform(-1e-3, 1e-3, (n, 3)),
    "mixed": lambda g, n: np.where(g.random((n, 3)) < 0.02, 1e3, 1.0) * g.uniform(-1, 1, (n, 3)),
    "far": lambda g, n: g.choice([-1, 1], (n, 3)) * 2.0 ** g.uniform(-40, 100, (n, 3)),
}


@pytest.fixture(scope="module")
def nrc():
    ctx = Context(0)
    m = Nrc(ctx, max_batch=64, seed=1)
    yield m
    m.close()
    ctx.close()


def _expose(features):
    """Parameters with which output k is input feature features[k]."""
    p = np.zeros(N.N_PARAMS, np.float32)
    W = [p[o:o + k * n].reshape(k, n) for o, (k, n) in zip(N.offsets(), N.LAYERS)]
    for j, f in enumerate(features):
        # neighbouring hidden units and ones of both chunks
        a, b = (j, j + 32)
        W[0][f, a], W[0][f, b] = 1.0, -1.0
        for w in W[1:5]:
            w[a, a] = w[b, b] = 1.0
        W[5][a, j], W[5][b, j] = 1.0, -1.0
    return p


def _exact(q):
    """FP64 features of the FP32 arguments, laid out as the network's inputs."""
    f = np.zeros((len(q), N.N_IN))
    for c in range(3):
        for k in range(12):
            a = (q[:, c] * np.float32(np.float32(np.pi) * np.float32(2.0 ** k))).astype(np.float64)
            f[:, 24 * c + 2 * k], f[:, 24 * c + 2 * k + 1] = np.sin(a), np.cos(a)
    f[:, 72:82] = q[:, 3:13]
    f[:, 82] = 1.0
    return f


@pytest.mark.parametrize("kind", list(POSITIONS))
def test_features(nrc, kind):
    g = np.random.default_rng(sum(map(ord, kind)))
    n = 1025   # whole tiles of 256 and one sample
    q = np.zeros((n, 13), np.float32)
    q[:, :3] = POSITIONS[kind](g, n)
    q[:, 3:] = g.normal(size=(n, 10))
    want = _exact(q)
    lo, hi = N.bf16(want - np.abs(want) * 2.0 ** -22), N.bf16(want + np.abs(want) * 2.0 ** -22)
    for first in range(0, 84, 3):
        fs = [f for f in range(first, first + 3) if f < 83]
        nrc.set_params(_expose(fs))
        got = nrc.infer(q)
        for j, f in enumerate(fs):
            bad = ~((got[:, j] >= lo[:, f]) & (got[:, j] <= hi[:, f]))
            assert not bad.any(), (f, int(bad.sum()), q[bad][0, :3], got[bad][0, j], want[bad][0, f])


def test_not_finite(nrc):
    """An infinite or NaN position gives NaN features, which the first layer's ReLU drops: the
    prediction is 0, as of a query whose hidden units are all off, and no other query's changes."""
    g = np.random.default_rng(7)
    q = g.random((300, 13)).astype(np.float32)
    nrc.set_params(_expose([0, 1, 30]))
    clean = nrc.infer(q)
    bad = q.copy()
    bad[::7, 0] = np.inf
    bad[3::7, 2] = np.nan
    got = nrc.infer(bad)
    hit = np.zeros(300, bool)
    hit[::7] = hit[3::7] = True
    np.testing.assert_array_equal(got[~hit], clean[~hit])
    np.testing.assert_array_equal(got[hit], 0.0)
