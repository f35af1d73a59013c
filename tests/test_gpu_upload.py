"""lg_segments_upload's bounds of the colours (the largest magnitude, whether all are >= 0), over the
values' bits: negative zero counts as zero, a NaN and an infinity as before, in either colour
array; and the keys it counts up."""
import numpy as np
import pytest

import light_garden_amd as lg

pytestmark = pytest.mark.gpu

BOUNDS = (-1.0, 1.0, -1.0, 1.0)


def image(ctx, pos, c0, c1=None):
    segs = lg.Segments(ctx, vertex_colors=c1 is not None)
    segs.upload(pos, c0, c1)
    np.testing.assert_array_equal(segs.download()[3], np.arange(len(pos), dtype=np.uint64))
    img = lg.Image(ctx, 192, 160, BOUNDS)
    img.accumulate(segs)
    return img.accum()


@pytest.mark.parametrize("n", [1, 63, 257, 1500])
@pytest.mark.parametrize("vertex", [False, True], ids=["one", "two"])
def test_colour_bounds(ctx, n, vertex):
    rng = np.random.default_rng(n)
    pos = rng.uniform(-1.0, 1.0, (n, 4)).astype(np.float32)
    c0 = rng.uniform(0.001, 0.02, (n, 4)).astype(np.float32)
    c1 = rng.uniform(0.001, 0.02, (n, 4)).astype(np.float32) if vertex else None
    last = c1 if vertex else c0
    last[-1, 1] = 0.0
    zero = image(ctx, pos, c0, c1)
    last[-1, 1] = -0.0
    np.testing.assert_array_equal(zero, image(ctx, pos, c0, c1))
    # a value below zero comes off the sums (two unsigned fields to a word could not hold that)
    last[:, 2] *= -1.0
    if vertex:
        c0[:, 2] *= -1.0
    below = image(ctx, pos, c0, c1)
    assert below[..., 2].min() < 0.0 or zero[..., 2].max() == 0.0
    np.testing.assert_allclose(below[..., 2], -zero[..., 2], rtol=1e-4, atol=1e-7)
    # a segment of NaN deposits nothing, and bounds nothing
    nan = np.full((1, 4), np.nan, np.float32)
    more = image(ctx, np.vstack([pos, pos[:1]]), np.vstack([c0, nan]), np.vstack([c1, nan]) if vertex else None)
    np.testing.assert_allclose(more, below, rtol=1e-5, atol=1e-8)
