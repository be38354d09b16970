"""Shadow rays through transparent surfaces, restarted by the lane that traces them: stacks of clear
panes between the scene and its sun, up to and beyond the 64 traces a ray gets, against the
oracle; the same images from a batch and (to rounding) from a two-level scene."""
import numpy as np
import pytest

from crender_amd import Context, Renderer, render_batch, scene_from_spec, scenes

pytestmark = pytest.mark.gpu
W, H, SPP, BOUNCES, SEED = 40, 24, 2, 2, 9


def _spec(panes):
    spec = scenes.sunlit(4, mode=1)
    n = len(spec.materials)
    spec.materials = list(spec.materials) + [scenes.MaterialSpec(colour=(0.9, 0.1, 0.1, 0.0))]
    tris = []
    for k in range(panes):   # 0.1 along the ray leaves a pane behind, not the next one
        y = 3.0 + 0.5 * k
        a, b, c, d = (-90.0, y, -90.0), (-90.0, y, 90.0), (90.0, y, 90.0), (90.0, y, -90.0)
        tris += [a, b, c, a, c, d]
    v = np.asarray(spec.vertices, np.float32).reshape(-1, 3)[np.asarray(spec.vertex_indices)]
    spec.vertices = np.concatenate([v, np.asarray(tris, np.float32).reshape(-1, 3)])
    spec.vertex_indices = np.arange(len(spec.vertices), dtype=np.uint32)
    spec.material_indices = np.concatenate([np.asarray(spec.material_indices, np.uint32),
                                            np.full(2 * panes, n, np.uint32)])
    spec.max_bounces, spec.rr_start = BOUNCES, 0
    return spec


def _render(ctx, sc):
    r = Renderer(ctx, sc, W, H, BOUNCES)
    r.set_resolution(W, H)
    r.set_options(mode=1, rr_start=0, seed=SEED)
    r.render(SPP)
    out, st = r.raw(), r.current_stats()
    r.close()
    return out, st


@pytest.mark.parametrize("stack", [8, 16, 32])
@pytest.mark.parametrize("panes", [0, 1, 5, 63, 64, 66])
def test_stacked_panes(oracle, panes, stack):
    spec = _spec(panes)
    ctx = Context(0, trace_stack=stack)
    sc = scene_from_spec(ctx, spec)
    got, st = _render(ctx, sc)
    ref = oracle.render(spec, res=(W, H), spp=SPP, seed=SEED, trav=oracle.BRUTE32)
    assert np.isclose(got, ref["raw"], rtol=1e-5, atol=1e-7).all(axis=2).mean() >= 0.995
    if panes < 64:   # every trace of a shadow ray counts
        assert abs(st["shadow_rays"] - ref["stats"]["shadow_rays"]) <= 0.005 * ref["stats"]["shadow_rays"]
    job = dict(scene=sc, width=W, height=H, spp=SPP, max_bounces=BOUNCES, mode=1, rr_start=0, seed=SEED)
    batch = render_batch(ctx, [job, job])[0]
    assert np.array_equal(batch[0], got) and np.array_equal(batch[1], got)
    sc.close()
    ctx.close()


def test_two_level_scene():
    spec = _spec(5)
    ctx = Context(0)
    sc = scene_from_spec(ctx, spec)
    flat, fst = _render(ctx, sc)
    one = np.eye(4, dtype=np.float32)
    far = one.copy()
    far[3, :3] = (0.0, -5000.0, 0.0)   # column-major: below everything
    sc.set_instances(0, [one.reshape(-1), far.reshape(-1)])
    sc.commit()
    two, tst = _render(ctx, sc)
    # the instance transform renormalises directions: equal but for rays that rounding sends elsewhere
    assert np.isclose(two, flat, rtol=1e-3, atol=1e-4).all(axis=2).mean() >= 0.95
    assert abs(tst["shadow_rays"] - fst["shadow_rays"]) <= 0.02 * fst["shadow_rays"]
    sc.close()
    ctx.close()
