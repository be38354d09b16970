"""Edges of the tiles of the post-processing and denoising kernels against the CPU restatements:
blur tiles of 64 x 32 pixels, a-trous tiles of 64 (steps 1 to 8) or 128 (step 16) pixels by 16
rows of a residue class, and the taps from global memory at steps above 16.

Bloom without a pow() is bit-exact; the denoiser keeps the bound of test_gpu_post.py.
"""
import numpy as np
import pytest

import post_oracle as P
from crender_amd import Context, denoise, post_process

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def _image(seed, h, w):
    img = np.random.default_rng(seed).random((h, w, 4), dtype=np.float32)
    img[..., :3] *= 1.5
    return img


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("h,w", [(1, 1), (8, 8), (9, 7), (31, 63), (32, 64), (33, 65), (46, 78), (65, 129), (70, 15)])
def test_bloom_tiles(ctx, h, w, full):
    img = _image(h * 131 + w, h, w)
    opts = dict(bloom=True, threshold=0.6, strength=0.7, tonemap=True, tonemap_type=2, full_coverage=full)
    assert np.array_equal(post_process(ctx, img, **opts), P.post_process(img, **opts))


@pytest.mark.parametrize("h,w,levels", [(1, 1, 1), (3, 5, 3), (16, 64, 1), (17, 65, 2), (20, 63, 5), (33, 129, 5),
                                        (130, 140, 5), (150, 70, 7)])
def test_atrous_tiles(ctx, h, w, levels):
    c, n, a = (_image(s + h, h, w) for s in (1, 2, 3))
    got = denoise(ctx, c, n, a, levels=levels)
    np.testing.assert_allclose(got, P.atrous(c, n, a, levels=levels), rtol=1e-4, atol=1e-5)


def test_atrous_infinite_pixel_stays_local(ctx):
    """An infinite colour makes its neighbours' sums non-finite only where it is a tap."""
    h, w = 40, 200
    c, n, a = (_image(s, h, w) for s in (4, 5, 6))
    want = denoise(ctx, c, n, a, levels=1)
    c[0, 0, :3] = np.inf
    got = denoise(ctx, c, n, a, levels=1)
    same = np.ones((h, w), bool)
    same[:3, :3] = False
    assert np.array_equal(got[same], want[same])


@pytest.mark.parametrize("which", ["colour", "normal", "albedo"])
def test_atrous_smallest_tolerances(ctx, which):
    """A tolerance whose inverse square is just finite lets no tap but the pixel's own and its equals
    through: an image without equal neighbours stays as it is."""
    h, w = 20, 70
    c, n, a = (_image(s, h, w) for s in (7, 8, 9))
    got = denoise(ctx, c, n, a, levels=1, **{f"sigma_{which}": 6e-20})
    np.testing.assert_allclose(got[..., :3], c[..., :3], rtol=3e-7)
