"""Deposits whose value overflows FP32 (an alpha above 1.8e19 squared; a colour times a factor): the
accumulator is infinite there, not zero. (Where channels share words, all of a scene's channels are
scaled for its largest value; hues have scales of their own, and keep their colours.) Every walk of frames that keep two channels per word: channels, runs, vertex colours, hues, blends with
factors, 32-pixel tiles; tiles of one item and split ones."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import abi, configs

pytestmark = pytest.mark.gpu

BOUNDS = (-1.0, 1.0, -1.0, 1.0)
BIG = 1e25


def check(got, ref, over, others):
    for c in over:
        deposited = ref[..., c] > 1e40  # (beyond FP32 by far)
        assert deposited.any() and np.isinf(got[..., c][deposited]).all()
        assert (got[..., c][ref[..., c] == 0.0] == 0.0).all()
    for c in others:
        assert np.abs(got[..., c] - ref[..., c]).sum() < 1e-4 * np.abs(ref[..., c]).sum()


@pytest.mark.parametrize("tuning", [{}, dict(min_piece=64, max_piece=256), dict(tile=32), dict(tile_block=512)],
                         ids=["default", "split", "tile32", "block512"])
@pytest.mark.parametrize("kind", ["channels", "runs", "vertex", "blend"])
def test_uploads(ctx, orc, kind, tuning):
    rng = np.random.default_rng(len(kind))
    n = 3000
    pos = rng.uniform(-1.0, 1.0, (n, 4)).astype(np.float32)
    col = np.full((n, 4), 0.25, np.float32) if kind == "runs" else rng.uniform(0.1, 1.0, (n, 4)).astype(np.float32)
    col[:, 3] *= BIG
    c1 = None
    if kind == "vertex":
        c1 = col[::-1].copy()
    if kind == "blend":
        col[:, 0] *= BIG
    segs = lg.Segments(ctx, vertex_colors=kind == "vertex")
    segs.upload(pos, col, c1)
    before = ctx.tuning()
    try:
        ctx.set_tuning(**tuning)
        img = lg.Image(ctx, 200, 150, BOUNDS)
        if kind == "blend":
            img.set_blend(color=(abi.BF_SRC, abi.BF_ONE, abi.BO_ADD))
        img.accumulate(segs)
        got = img.accum().astype(np.float64)
    finally:
        ctx.set_tuning(**before)
    view = abi.LgView(*BOUNDS, 200, 150)
    ref = orc.accumulate_f64(pos.astype(np.float64), col, c1, view, threads=8)
    if kind == "blend":
        ref[..., 0] *= BIG  # (of about the size: the reference deposits the colour once)
    check(got, ref, (0, 3) if kind == "blend" else (3,), ())


@pytest.mark.parametrize("n_lights", [1, 2, 4])
def test_traced(ctx, orc, n_lights):
    scene = configs.plain_small(2000)
    tr = lg.Tracer(ctx, scene.canvas)
    for o in scene.objects:
        tr.push_object(o)
    for k in range(n_lights):
        tr.push_light(lg.PointLight((0.05 + 0.1 * k, 0.02), 1500, [0.5, 1.0, 0.25, BIG]))
    tr.cutoff_color = [0.0] * 4
    segs, img = lg.Segments(ctx), lg.Image(ctx, 200, 150, BOUNDS)
    tr.render(segs, img)
    pos, col, _, _ = segs.download()
    ref = orc.accumulate_f64(pos.astype(np.float64), col, None, abi.LgView(*BOUNDS, 200, 150), threads=8)
    check(img.accum().astype(np.float64), ref, (3,), (0, 1, 2) if n_lights < 4 else ())
