"""4-wide trees: overlapping triangles of common axis-aligned planes, every one there three times, each in a leaf
of its own: the closest hit is that of the CPU oracle's brute force, the smallest primID of the
triangles at the smallest distance, whichever the order of the walk.

A triangle in a face of its box has a hit distance that rounds apart from the face's.  The rays
meet the planes at 3 degrees and more, where the two differ by less than 2^-16 relative (FP32
roundings of a few units in the last place over the sine of the angle), a sixteenth of what
the 4-wide traversal allows for.
"""
import numpy as np
import pytest

from crender_amd import Context, scene_from_spec, scenes

pytestmark = pytest.mark.gpu


def _planes(seed, n=240):
    rng = np.random.default_rng(seed)
    v = rng.uniform(-1, 1, (n, 3, 3)).astype(np.float32)
    axis, height = rng.integers(0, 3, n), rng.choice([-0.7, -0.31, 0.123, 0.55], n).astype(np.float32)
    for k in range(n):
        v[k, :, axis[k]] = height[k]
    return np.repeat(v, 3, axis=0)[rng.permutation(3 * n)]


def test_coplanar_and_coincident_4_wide(oracle):
    tri = _planes(3)
    n = len(tri)
    spec = scenes.soup(n, seed=1)
    spec.vertices = tri.reshape(-1, 3)
    spec.vertex_indices = np.arange(3 * n, dtype=np.uint32)
    ctx = Context(0, bvh_width=4, max_leaf=1)
    sc = scene_from_spec(ctx, spec)
    rng = np.random.default_rng(4)
    m = 40_000
    o = rng.uniform(-3, 3, (m, 3)).astype(np.float32)
    d = rng.uniform(-1, 1, (m, 3)).astype(np.float32) - o
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    keep = np.abs(d).min(1) > 0.0524
    o, d = o[keep], d[keep]
    assert len(o) > 20_000
    got = sc.cast_rays(o, d)
    p32, t32, _, _ = oracle.intersect(tri.reshape(n, 9), o, d, oracle.BRUTE32)
    gp = got["prim_id"].astype(np.int64)
    gp[gp == 0xFFFFFFFF] = -1
    assert (p32 >= 0).mean() > 0.5
    assert np.array_equal(gp, p32), int((gp != p32).sum())
    hit = p32 >= 0
    assert np.array_equal(got["t"][hit], t32[hit].astype(np.float32))
    ctx.close()
