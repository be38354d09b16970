"""Ray counts at the edges of the traversal's work distribution (RaySupply in traverse.hip).

The queue is cut into 8 slices; a wave owns 64 rays of its slice by position and the rest of
a slice is handed out in chunks.  The counts cover slices that are empty, not full or one ray
long, blocks without rays, exactly the rays owned by position (256 CUs x 2 blocks x 4 waves x
64 = 131,072), one ray more or less (one chunk of one ray per slice, slices of unequal
length), and several chunks per wave.  Every ray's hit equals the FP32 oracle's, bit for bit.
"""
import numpy as np
import pytest

from crender_amd import Context, scene_from_spec, scenes

pytestmark = pytest.mark.gpu

OWNED = 131_072


@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 64, 65, 511, 513, 2047, 2049, OWNED - 1, OWNED, OWNED + 1, OWNED + 9,
                               3 * OWNED + 5])
def test_every_ray_is_traced_once(oracle, n):
    spec = scenes.cornell(1)
    ctx = Context(0)
    sc = scene_from_spec(ctx, spec)
    o, d = scenes.diffuse_rays(n, seed=n, lo=-0.9, hi=0.9)
    o[:, 1] += 1.0
    got = sc.cast_rays(o, d)
    occ = sc.occluded(o, d, tfar=0.75)
    sc.close()
    ctx.close()
    p, t, u, v = oracle.intersect(spec.corners(), o, d, oracle.BRUTE32)
    gp = got["prim_id"].astype(np.int64)
    gp[gp == 0xFFFFFFFF] = -1
    assert np.array_equal(gp, p)
    hit = p >= 0
    assert np.array_equal(got["t"][hit], t[hit].astype(np.float32)) and np.all(np.isinf(got["t"][~hit]))
    assert np.array_equal(got["u"][hit], u[hit].astype(np.float32))
    assert np.array_equal(got["v"][hit], v[hit].astype(np.float32))
    assert np.array_equal(occ, hit & (t.astype(np.float32) <= np.float32(0.75)))
