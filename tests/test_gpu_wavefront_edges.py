"""Edges of the wavefront kernels' launches: images smaller and larger than a block, wavefronts
of one to eight passes (accumulation through LDS), and more paths than the shading grid has
threads (2,560 blocks of 256), where its blocks loop.  Images equal the oracle's bit for bit, and
those of launch shapes in which nothing loops."""
import numpy as np
import pytest

from crender_amd import Context, Renderer, render_batch, scene_from_spec, scenes

pytestmark = pytest.mark.gpu


def _render(spec, w, h, bounces, spp, mode, **kw):
    ctx = Context(0, **kw)
    sc = scene_from_spec(ctx, spec)
    r = Renderer(ctx, sc, w, h, bounces)
    r.set_resolution(w, h)
    r.set_options(mode=mode, rr_start=3, seed=11)
    r.render(spp)
    out = r.raw()
    r.close()
    sc.close()
    ctx.close()
    return out


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("w,h,spp", [(1, 1, 8), (17, 15, 7), (16, 16, 3), (257, 1, 5), (33, 31, 9)])
def test_small_images(oracle, w, h, spp, mode):
    spec = scenes.sunlit(4, mode=mode)
    spec.max_bounces, spec.rr_start = 5, 3
    got = _render(spec, w, h, 5, spp, mode)
    assert np.array_equal(got, _render(spec, w, h, 5, spp, mode, wavefront_paths=1))   # one pass at a time
    ref = oracle.render(spec, res=(w, h), spp=spp, seed=11, trav=oracle.BRUTE32)["raw"]
    assert np.array_equal(got, ref)


def test_more_paths_than_shading_threads(oracle):
    spec = scenes.cornell(1)
    spec.max_bounces, spec.rr_start = 2, 3
    w, h = 1024, 650   # 665,600 paths
    got = _render(spec, w, h, 2, 1, 0)
    # the same paths 131,072 at a time
    ctx = Context(0)
    job = dict(scene=scene_from_spec(ctx, spec), width=w, height=h, spp=1, max_bounces=2, mode=0, rr_start=3, seed=11)
    chunks, _, stats = render_batch(ctx, [job], max_paths=131_072)
    assert stats["replays"] == 6 and np.array_equal(got, chunks[0])
    ctx.close()
    ref = oracle.render(spec, res=(w, h), spp=1, seed=11, trav=oracle.BRUTE32)["raw"]
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("spp", [7, 8])
def test_lone_wavefront_in_halves(spp):
    spec = scenes.sunlit(4, mode=1)
    w, h = 1536, 1024   # 8 passes are 12,582,912 paths, the fewest that are split
    got = _render(spec, w, h, 2, spp, 1)
    assert np.array_equal(got, _render(spec, w, h, 2, spp, 1, wavefront_paths=w * h))   # a pass at a time
