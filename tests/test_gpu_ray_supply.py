"""Ray counts at the edges of the traversal's work distribution (RaySupply in traverse.hip).

The queue is cut into 8 slices; a wave owns 64 rays of its slice by position and the rest of
a slice is handed out in chunks.  The counts cover slices that are empty, not full or one ray
long, blocks without rays, exactly the rays owned by position, one ray more or less (one chunk
of one ray per slice, slices of unequal length), and several chunks per wave, for the grid of
crt_intersect (256 CUs x 4 blocks x 4 waves x 64 = 262,144 rays owned; it traces up to 65,536
rays with eight lanes per ray instead) and that of crt_intersect_noalloc (64 blocks, 16,384
rays owned, a ray per lane at every count).  Every ray's hit equals the FP32 oracle's, bit for bit.
"""
import numpy as np
import pytest

from _devmem import DeviceArrays
from crender_amd import Context, scene_from_spec, scenes

pytestmark = pytest.mark.gpu

OWNED, OWNED_NOALLOC = 262_144, 16_384
KEYS = ("org_x", "org_y", "org_z", "dir_x", "dir_y", "dir_z", "tnear", "tfar")


def _check(oracle, spec, o, d, got):
    p, t, u, v = oracle.intersect(spec.corners(), o, d, oracle.BRUTE32)
    gp = got["prim_id"].astype(np.uint32).astype(np.int64)
    gp[gp == 0xFFFFFFFF] = -1
    assert np.array_equal(gp, p)
    hit = p >= 0
    assert np.array_equal(got["t"][hit], t[hit].astype(np.float32)) and np.all(np.isinf(got["t"][~hit]))
    assert np.array_equal(got["u"][hit], u[hit].astype(np.float32))
    assert np.array_equal(got["v"][hit], v[hit].astype(np.float32))
    return hit, t.astype(np.float32)


def _rays(n):
    o, d = scenes.diffuse_rays(n, seed=n, lo=-0.9, hi=0.9)
    o[:, 1] += 1.0
    return o, d


@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 64, 65, 511, 513, 65_536, 65_537, 98_304, 98_305, OWNED - 1, OWNED, OWNED + 1,
                               OWNED + 9, 2 * OWNED + 5])
def test_every_ray_is_traced_once(oracle, n):
    spec = scenes.cornell(1)
    ctx = Context(0)
    sc = scene_from_spec(ctx, spec)
    o, d = _rays(n)
    got = sc.cast_rays(o, d)
    occ = sc.occluded(o, d, tfar=0.75)
    sc.close()
    ctx.close()
    hit, t = _check(oracle, spec, o, d, got)
    assert np.array_equal(occ, hit & (t <= np.float32(0.75)))


@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 64, 65, 511, 513, 2047, 2049, OWNED_NOALLOC - 1, OWNED_NOALLOC,
                               OWNED_NOALLOC + 1, OWNED_NOALLOC + 9, 5 * OWNED_NOALLOC + 3])
def test_every_ray_is_traced_once_on_the_small_grid(oracle, n):
    spec = scenes.cornell(1)
    ctx = Context(0)
    sc = scene_from_spec(ctx, spec)
    o, d = _rays(n)
    dev = DeviceArrays()
    cols = [o[:, 0], o[:, 1], o[:, 2], d[:, 0], d[:, 1], d[:, 2], np.full(n, 1e-5), np.full(n, np.inf)]
    types = dict(t=np.float32, u=np.float32, v=np.float32, prim_id=np.uint32)
    out = {k: dev.put(np.zeros(n, dt)) for k, dt in types.items()}
    sc.cast_rays_device({k: dev.put(np.asarray(c, np.float32)) for k, c in zip(KEYS, cols)}, out, n, noalloc=True)
    got = {k: dev.get(out[k], n, dt) for k, dt in types.items()}
    dev.free()
    sc.close()
    ctx.close()
    _check(oracle, spec, o, d, got)
