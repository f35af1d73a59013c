"""Accumulation of segments in runs of one colour (StringMods without modulo colours): one weight plane
per run, colours applied to the sums. Sizes where it can go wrong: one run, a full layer of six, a
layer of one after it, the most runs (four layers) and one more (which takes the walk by colours),
neighbours of equal colour, a colour of zero, lists split over many work items, frames of more than
8192 tiles' scan, another blend. Against the FP64 accumulation of the same segments, within the
bound that the walk by colours keeps, and bit for bit over tunings, a repeated call and
lg_accumulate_noalloc."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import abi, string_mod

pytestmark = pytest.mark.gpu

BOUNDS = (-1.0, 1.0, -1.0, 1.0)


def drawn(ctx, n_mods, points, rng):
    colors = [[float(x) for x in rng.uniform(0.0002, 0.004, 4)] for _ in range(n_mods)]
    if n_mods > 2:
        colors[1] = [0.0, 0.0, 0.0, 0.0]
        colors.insert(2, list(colors[2]))  # two neighbours of one colour: one run
    segs = lg.Segments(ctx, vertex_colors=True)
    string_mod.draw(ctx, [lg.StringMod(modulo=points + 7 * i, num=2 + 3 * i, scale=0.93, color=c)
                          for i, c in enumerate(colors)], segs)
    return segs


def accumulated(ctx, segs, w, h, blend=None, noalloc=False, **tuning):
    before = ctx.tuning()
    try:
        ctx.set_tuning(**tuning)
        img = lg.Image(ctx, w, h, BOUNDS)
        if blend:
            img.set_blend(color=blend)
        if noalloc:
            img.accumulate_noalloc(segs)
        else:
            img.accumulate(segs)
        return img.accum()
    finally:
        ctx.set_tuning(**before)


@pytest.mark.parametrize("n_mods,points,w,h", [(1, 900, 640, 480), (6, 1500, 500, 701), (7, 1500, 1024, 64),
                                               (24, 400, 333, 333), (25, 400, 333, 333)])
def test_runs_equal_fp64_accumulation(ctx, orc, n_mods, points, w, h):
    segs = drawn(ctx, n_mods, points, np.random.default_rng(n_mods))
    got = accumulated(ctx, segs, w, h)
    pos, c0, _, _ = segs.download()
    ref = orc.accumulate_f64(pos.astype(np.float64), c0, None, abi.LgView(*BOUNDS, w, h), threads=8)
    e = orc.rel_l1(got, ref)
    ea = np.abs(got[..., 3] - ref[..., 3]).sum() / np.abs(ref[..., 3]).sum()
    print("%d StringMods: rel L1 %.3e (alpha %.3e)" % (n_mods, e, ea))
    assert e < 1e-5 and ea < 1e-5
    for tuning in (dict(min_piece=64, max_piece=64), dict(tile_block=512), dict(min_piece=64, max_piece=1 << 20), {}):
        np.testing.assert_array_equal(got, accumulated(ctx, segs, w, h, **tuning))
    np.testing.assert_array_equal(got, accumulated(ctx, segs, w, h, noalloc=True))


def test_runs_other_blend_and_large_image(ctx, orc):
    segs = drawn(ctx, 7, 500, np.random.default_rng(3))
    pos, c0, _, _ = segs.download()
    got = accumulated(ctx, segs, 512, 512, blend=(abi.BF_SRC_ALPHA, abi.BF_ONE, abi.BO_ADD))
    col = c0.copy()
    col[:, :3] *= c0[:, 3:]
    ref = orc.accumulate_f64(pos.astype(np.float64), col, None, abi.LgView(*BOUNDS, 512, 512), threads=8)
    assert orc.rel_l1(got, ref) < 1e-5
    w, h = 6464, 6016  # 101 x 94 tiles: the multi-block scan
    got = accumulated(ctx, segs, w, h)
    np.testing.assert_array_equal(got, accumulated(ctx, segs, w, h, min_piece=64, max_piece=64))
    ref = orc.accumulate_f64(pos.astype(np.float64), c0, None, abi.LgView(*BOUNDS, w, h), threads=8)
    assert orc.rel_l1(got, ref) < 1e-5


@pytest.mark.parametrize("far", [1e6, 1e15, 1e18], ids=lambda f: "%.0e" % f)
def test_runs_of_far_end_points(ctx, far):
    """Lines across the image from far outside (FP32 end points, so they come from anywhere in it): the
    tiles of the walk by weights and of the walk by colours hold the same amount."""
    rng = np.random.default_rng(int(np.log10(far)))
    n = 4000
    a = rng.uniform(0.0, 2 * np.pi, n)
    c = rng.uniform(-1.0, 1.0, (n, 2))
    d = np.stack([np.cos(a), np.sin(a)], 1) * far
    pos = np.concatenate([c - d, c + d], 1).astype(np.float32)
    col = np.full((n, 4), 0.002, np.float32)
    runs, colours = lg.Segments(ctx), lg.Segments(ctx)
    runs.upload(pos, col)
    col2 = col.copy()
    col2[::2] *= np.float32(1.0 + 2.0 ** -20)  # (a run each: the walk by colours)
    colours.upload(pos, col2)
    x, y = accumulated(ctx, runs, 512, 512), accumulated(ctx, colours, 512, 512)
    assert np.isfinite(x).all()
    np.testing.assert_allclose(x.sum(), y.sum(), rtol=1e-3)
