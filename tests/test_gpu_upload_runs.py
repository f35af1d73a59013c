"""Uploads find their runs of one colour by stretches of 256 colours: the image against the FP64
accumulation with the colour changing around a stretch's end, at the last segment and within one, and
with the most runs (24) and one more; and an upload of one colour takes about as long as one
whose colours all differ (which has no runs to find)."""
import time

import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import abi

pytestmark = pytest.mark.gpu

BOUNDS = (-1.0, 1.0, -1.0, 1.0)


def at_every(k, n_runs):
    return [k * i for i in range(1, n_runs)]


@pytest.mark.parametrize("n,changes", [(1700, [255]), (1700, [256]), (1700, [257, 258]), (30000, [1, 511, 512, 513, 1699]), (1700, []),
                                       (257, [256]), (500000, at_every(1000, 24)), (2500, at_every(100, 25))],
                         ids=lambda v: str(len(v)) if isinstance(v, list) else str(v))
def test_runs_around_stretches(ctx, orc, n, changes):
    rng = np.random.default_rng(n + len(changes))
    pos = rng.uniform(-1.0, 1.0, (n, 4)).astype(np.float32)
    bounds = [0] + changes + [n]
    col = np.empty((n, 4), np.float32)
    for k, (a, b) in enumerate(zip(bounds, bounds[1:])):
        col[a:b] = rng.uniform(0.001, 0.01, 4) * (1.0 + 9.0 * (k % 2))
    segs = lg.Segments(ctx)
    segs.upload(pos, col)
    img = lg.Image(ctx, 300, 200, BOUNDS)
    img.accumulate(segs)
    ref = orc.accumulate_f64(pos.astype(np.float64), col, None, abi.LgView(*BOUNDS, 300, 200), threads=8)
    assert orc.rel_l1(img.accum(), ref) < 1e-5


def test_one_colour_uploads_take_no_longer(ctx):
    rng = np.random.default_rng(1)
    n = 400000
    pos = rng.uniform(-1.0, 1.0, (n, 4)).astype(np.float32)
    many = rng.uniform(0.001, 0.01, (n, 4)).astype(np.float32)
    one = np.full((n, 4), 0.002, np.float32)
    segs = lg.Segments(ctx, capacity=n)
    best = {}
    for _ in range(40):
        for name, col in (("many", many), ("one", one)):
            t = time.perf_counter()
            segs.upload(pos, col)
            best[name] = min(best.get(name, 1.0), time.perf_counter() - t)
    print("one colour %.0f us, all different %.0f us" % (1e6 * best["one"], 1e6 * best["many"]))
    assert best["one"] < 1.4 * best["many"]
