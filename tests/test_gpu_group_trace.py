"""Small batches, traced with eight lanes per ray, against the same rays as part of a batch large
enough for a ray per lane (more than 65,536 rays): every field is equal.  Scenes with leaves of
up to 16 triangles, coincident triangles (ties go to the smaller primID) and deep trees; rays
with limits that cut hits off, degenerate and non-finite rays."""
import numpy as np
import pytest

from crender_amd import Context, scene_from_spec, scenes

pytestmark = pytest.mark.gpu

LARGE = 100_000


def _rays(n, seed):
    o, d = scenes.diffuse_rays(n, seed=seed)
    rng = np.random.default_rng(seed)
    d = (d * rng.uniform(0.2, 3.0, (n, 1))).astype(np.float32)
    tn = np.where(rng.random(n) < 0.2, 0.1, 1e-5).astype(np.float32)
    tf = np.where(rng.random(n) < 0.3, 0.2, np.inf).astype(np.float32)
    if n >= 16:
        d[0] = 0.0                       # no direction
        d[1] = (0.0, 0.0, 1.0)           # axis-parallel
        d[2] = (0.0, -1.0, 0.0)
        o[3, 0] = np.nan
        tn[4], tf[4] = 0.5, 0.1          # empty interval
        tf[5] = np.nan
        d[6] = (np.inf, 1.0, 0.0)
        o[7] = (1e30, 0.0, 0.0)
    return o, d, tn, tf


def _coincident():
    spec = scenes.soup(300, seed=3, sigma=0.2)
    v = spec.vertices.reshape(-1, 3, 3).copy()
    v[40:80] = v[40]
    v[100:108] = v[100]
    spec.vertices = v.reshape(-1, 3)
    return spec


SCENES = {"soup": (lambda: scenes.soup(30_000, seed=8, sigma=0.02), {}),
          "fuller leaves": (lambda: scenes.soup(3_000, seed=9, sigma=0.05), dict(max_leaf=16, bvh_prim_cost=0.05)),
          "coincident": (_coincident, dict(max_leaf=16, bvh_prim_cost=0.05)),
          "one triangle": (lambda: scenes.soup(1, seed=2, sigma=0.4), {}),
          "terrain": (lambda: scenes.terrain(grid=128, spheres=30, seed=5), {})}


@pytest.mark.parametrize("stack", [8, 16, 32])
@pytest.mark.parametrize("name", SCENES)
def test_group_equals_lane(name, stack):
    make, kw = SCENES[name]
    ctx = Context(0, trace_stack=stack, **kw)
    sc = scene_from_spec(ctx, make())
    n = 4_099
    o, d, tn, tf = _rays(n, 21)
    rep = LARGE // n + 1
    big = [np.tile(x, (rep, 1) if x.ndim == 2 else rep) for x in (o, d, tn, tf)]
    lane = sc.cast_rays(*big, normals=True)
    rec = sc.cast_ray_records(*big)
    occ = sc.occluded(*big)
    for m in (1, 9, 33, n):
        got = sc.cast_rays(o[:m], d[:m], tn[:m], tf[:m], normals=True)
        for k, v in got.items():
            assert np.array_equal(v, lane[k][:m], equal_nan=True), (k, m)
        got = sc.cast_ray_records(o[:m], d[:m], tn[:m], tf[:m])
        for k, v in got.items():
            assert np.array_equal(v, rec[k][:m], equal_nan=True), (k, m)
        assert np.array_equal(sc.occluded(o[:m], d[:m], tn[:m], tf[:m]), occ[:m])
    sc.close()
    ctx.close()
