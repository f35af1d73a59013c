"""Traced segments as hues (a segment's colour is its light's, scaled): one LDS word per deposit, two
samples to a lane. One to three lights take it, four do not; a frame beside a scene with negative
colours walks hues pair by pair. Against the FP64 accumulation of the same segments, and bit for bit
between the walks, pieces of any size and lg_accumulate_noalloc."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import abi, configs

pytestmark = pytest.mark.gpu

CANVAS = (-1.0, 1.0, -1.0, 1.0)


def tracer(ctx, colors, rays):
    tr = lg.Tracer(ctx, CANVAS)
    for o in configs.large_single(num_rays=1, width=64).objects[:9]:
        tr.push_object(o)
    for k, c in enumerate(colors):
        tr.push_light(lg.PointLight((-0.8 + 0.4 * k, 0.31 - 0.2 * k), rays + 7 * k, c))
    tr.max_bounce = 5
    return tr


def lights(n):
    rng = np.random.default_rng(n)
    c = [[float(x) for x in rng.uniform(0.001, 0.02, 4)] for _ in range(n)]
    c[0] = [0.01, 0.0, 0.0, 0.01]  # one channel only
    return c


@pytest.mark.parametrize("n,rays,side", [(1, 1, 65), (1, 900, 511), (2, 2000, 640), (3, 3000, 512), (4, 1500, 512)])
def test_hues_equal_fp64_accumulation_and_each_other(ctx, orc, n, rays, side):
    def rendered(**tuning):
        before = ctx.tuning()
        try:
            ctx.set_tuning(**tuning)
            img = lg.Image(ctx, side, side, CANVAS)
            img.accumulate(segs)
            return img.accum()
        finally:
            ctx.set_tuning(**before)

    tr = tracer(ctx, lights(n), rays)
    segs = tr.trace()
    pos, c0, _, _ = segs.download()
    got = rendered()
    ref = orc.accumulate_f64(pos.astype(np.float64), c0, None, abi.LgView(*CANVAS, side, side), threads=8)
    e = orc.rel_l1(got, ref)
    ea = np.abs(got[..., 3] - ref[..., 3]).sum() / np.abs(ref[..., 3]).sum()
    print("%d lights: rel L1 %.3e (alpha %.3e)" % (n, e, ea))
    assert e < 1e-5 and ea < 1e-5
    np.testing.assert_array_equal(got, rendered(min_piece=64, max_piece=64))
    img = lg.Image(ctx, side, side, CANVAS)
    img.accumulate_noalloc(segs)
    np.testing.assert_array_equal(got, img.accum())


def test_hues_beside_a_scene_with_negative_colours(ctx):
    a, b = tracer(ctx, lights(3), 2500), tracer(ctx, [[-0.01, 0.02, 0.01, 0.5]], 700)
    alone, both, other = (lg.Image(ctx, 512, 512, CANVAS) for _ in range(3))
    lg.batch_render(ctx, [a], [lg.Segments(ctx)], [alone])
    lg.batch_render(ctx, [a, b], [lg.Segments(ctx), lg.Segments(ctx)], [both, other])
    # (the order of a trace's segments changes no bit of the sums)
    np.testing.assert_array_equal(alone.accum(), both.accum())
    assert other.accum()[..., 0].min() < 0.0
