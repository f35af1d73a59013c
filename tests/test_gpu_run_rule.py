"""Which accumulations sum weights of runs of one colour: those whose samples save more than the runs'
planes and layers cost. Both sides of the rule against the FP64 accumulation, with the walk that was
taken read off its LDS atomics; several layers, work split and lg_accumulate_noalloc bit for bit; and
an upload in many runs takes no longer than one whose colours all differ."""
import time

import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import abi, string_mod

pytestmark = pytest.mark.gpu

BOUNDS = (-1.0, 1.0, -1.0, 1.0)


def accumulated(ctx, segs, w, h, noalloc=False, **tuning):
    """The accumulator, and whether weights were summed: 4 atomics to a step of up to 128 samples, by
    channels 8."""
    before = ctx.tuning()
    img = lg.Image(ctx, w, h, BOUNDS)
    try:
        ctx.set_tuning(**tuning)
        ctx.set_profiling(True)
        (img.accumulate_noalloc if noalloc else img.accumulate)(segs)
        _, _, samples, atomics = ctx.stage_times().get("tile_accum", (0, 0, 0, 0))
        return img.accum(), bool(samples) and 64.0 * atomics / samples < 3.9
    finally:
        ctx.set_profiling(False)
        ctx.set_tuning(**before)
        img.close()


def lines(ctx, n, runs, length, seed=0):
    rng = np.random.default_rng(seed)
    c, a = rng.uniform(-0.9, 0.9, (n, 2)), rng.uniform(0.0, 2 * np.pi, n)
    d = np.stack([np.cos(a), np.sin(a)], 1) * 0.5 * length
    pos = np.concatenate([c - d, c + d], 1).astype(np.float32)
    col = np.repeat(rng.uniform(0.0005, 0.004, (runs, 4)).astype(np.float32), -(-n // runs), axis=0)[:n]
    segs = lg.Segments(ctx)
    segs.upload(pos, col)
    return segs, pos, col


@pytest.mark.parametrize("n,runs,length,w,h,weights", [
    (300, 3, 0.01, 700, 500, None), (300, 4, 0.01, 700, 500, None), (60000, 6, 1.0, 500, 701, True),
    (120000, 7, 1.2, 256, 256, True), (120000, 7, 0.01, 256, 256, False), (250000, 13, 1.2, 512, 400, True),
    (700000, 24, 1.2, 320, 256, True), (50000, 24, 0.02, 1024, 1024, False)])
def test_both_sides_of_the_rule(ctx, orc, n, runs, length, w, h, weights):
    segs, pos, col = lines(ctx, n, runs, length)
    got, by_weights = accumulated(ctx, segs, w, h)
    assert weights is None or by_weights == weights  # (few samples leave a step's lanes empty)
    ref = orc.accumulate_f64(pos.astype(np.float64), col, None, abi.LgView(*BOUNDS, w, h), threads=8)
    assert orc.rel_l1(got, ref) < 1e-5
    for tuning in (dict(min_piece=64, max_piece=4096), dict(min_piece=64, max_piece=1 << 20)):
        np.testing.assert_array_equal(got, accumulated(ctx, segs, w, h, **tuning)[0])
    np.testing.assert_array_equal(got, accumulated(ctx, segs, w, h, noalloc=True)[0])


def test_generated_and_uploaded_take_one_walk(ctx):
    for points, weights in ((400, False), (60000, True)):
        rng = np.random.default_rng(points)
        mods = [lg.StringMod(modulo=points, num=2 + i, scale=0.9, color=[float(x) for x in rng.uniform(0.001, 0.004, 4)])
                for i in range(8)]
        drawn, up = lg.Segments(ctx, vertex_colors=True), lg.Segments(ctx)
        string_mod.draw(ctx, mods, drawn)
        pos, col, _, _ = drawn.download()
        up.upload(pos, col)
        (a, wa), (b, wb) = accumulated(ctx, drawn, 256, 256), accumulated(ctx, up, 256, 256)
        assert wa == wb == weights
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("runs", [7, 24])
def test_runs_take_no_longer_than_channels(ctx, runs):
    n = 25000
    few, pos, col = lines(ctx, n, runs, 0.002)
    many = lg.Segments(ctx)
    col2 = col.copy()
    col2[::3] *= np.float32(1.0 + 2.0 ** -20)
    many.upload(pos, col2)
    img = lg.Image(ctx, 4096, 4096, BOUNDS)
    best = {}
    for _ in range(40):
        for name, segs in (("runs", few), ("channels", many)):
            t = time.perf_counter()
            img.accumulate(segs)
            best[name] = min(best.get(name, 1.0), time.perf_counter() - t)
    print("%d runs %.0f us, all different %.0f us" % (runs, 1e6 * best["runs"], 1e6 * best["channels"]))
    assert best["runs"] < 1.15 * best["channels"]
