"""What a segment buffer holds after a call on it failed: the old segments where the call was refused
before it touched them, none where the frame had begun to overwrite them. Either way the buffer is
good for any later call: its counts, its rays and its FP64 end points describe what is in it."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import abi, configs
from light_garden_amd import geo as G

pytestmark = pytest.mark.gpu

BOUNDS = (-1.0, 1.0, -1.0, 1.0)


def tracer(ctx, scene, fp64=False):
    tr = lg.Tracer(ctx, scene.canvas)
    for o in scene.objects:
        tr.push_object(o)
    for l in scene.lights:
        tr.push_light(l)
    tr.max_bounce = scene.max_bounce
    tr.cutoff_color = list(scene.cutoff)
    tr.fp64 = fp64
    return tr


def same(a, b):
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])


@pytest.mark.parametrize("fp64", [False, True], ids=["fp32", "fp64"])
def test_refused_frames_leave_the_segments(ctx, fp64):
    segs = lg.Segments(ctx)
    tr = tracer(ctx, configs.plain_small(500), fp64)
    want = tr.trace(segs).vertices()
    # more FP64 records than the trace holds on chip, and more rays than the buffer has room for
    rng = configs.SplitMix64(1)
    big = tracer(ctx, configs.Scene(configs.random_objects(rng, 640), [lg.PointLight((0.0, 0.0), 50000, [1.0] * 4)]), True)
    with pytest.raises(abi.LgError, match="too large"):
        big.trace(segs)
    same(segs.vertices(), want)
    # an image with more tiles than the binning counts
    more = tracer(ctx, configs.plain_small(50000))
    img = lg.Image(ctx, 8192, 4160, BOUNDS)
    before = ctx.tuning()
    try:
        ctx.set_tuning(tile=32)
        with pytest.raises(abi.LgError, match="4096x4096"):
            more.render(segs, img)
    finally:
        ctx.set_tuning(**before)
    same(segs.vertices(), want)
    if fp64:
        assert segs.download_pos64().shape == (segs.count(), 4)
    img.close()


def test_failed_frame_leaves_no_segments(ctx):
    """A frame of more than 2^32 segment-tile pairs fails after its trace has overwritten the buffer with the
    segments of other, more rays."""
    def corner_light(n, flip):
        a, b = (-0.9, -0.99), (-0.99, -0.9)
        return [lg.DirectionalLight([0.01] * 4, n, G.LineSegment(b, a) if flip else G.LineSegment(a, b))]

    segs = lg.Segments(ctx)
    flip = False
    for flip in (False, True):  # the one that shines along the image's diagonal
        pos = tracer(ctx, configs.Scene([], corner_light(100, flip), max_bounce=1)).trace(segs).download()[0]
        if np.hypot(pos[:, 2] - pos[:, 0], pos[:, 3] - pos[:, 1]).mean() > 2.0:
            break
    else:
        pytest.fail("neither light crosses the image")
    small = tracer(ctx, configs.plain_small(300), True)
    want = small.trace(segs).vertices()
    many = tracer(ctx, configs.Scene([], corner_light(20_000_000, flip), max_bounce=1))
    img = lg.Image(ctx, 4096, 4096, BOUNDS)
    before = ctx.tuning()
    try:
        ctx.set_tuning(tile=32)
        with pytest.raises(abi.LgError, match="2\\^32"):
            many.render(segs, img)
    finally:
        ctx.set_tuning(**before)
    many.close()
    assert segs.count() == 0
    xy, rgba = segs.vertices()
    assert xy.shape == (0, 2) and rgba.shape == (0, 4)
    with pytest.raises(abi.LgError):
        segs.download_pos64()
    img.clear()
    img.accumulate(segs)
    assert not img.accum().any()
    # and the buffer takes a trace again
    small.trace(segs)
    same(segs.vertices(), want)
    assert segs.download_pos64().shape == (segs.count(), 4)
    img.close()
    segs.close()
