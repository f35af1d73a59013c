"""How the tiles' lists are cut: where the tile kernel walks pair by pair (32-pixel tiles; one channel per
word), the default pieces leave no workgroup far behind the others, as pieces of at most 8192 pairs
do not; images are the same bits for either."""
import time

import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import string_mod

pytestmark = pytest.mark.gpu

BOUNDS = (-1.0, 1.0, -1.0, 1.0)


@pytest.mark.parametrize("tuning", [dict(tile=32), dict(tile_block=512), {}], ids=["tile32", "block512", "default"])
@pytest.mark.parametrize("packed", [True, False], ids=["two_channels", "one_channel"])
def test_default_pieces(ctx, packed, tuning):
    rng = np.random.default_rng(4)
    colors = lambda: [float(x) for x in rng.uniform(0.0005, 0.004, 4)]
    mods = [lg.StringMod(modulo=48074, num=2 + i, scale=0.9, color=colors(), modulo_colors=[string_mod.ModRemColor(3, 1, colors())])
            for i in range(16)]
    segs = lg.Segments(ctx, vertex_colors=True)
    string_mod.draw(ctx, mods, segs)
    before = ctx.tuning()
    best, images = {}, {}
    try:
        ctx.set_packed_accumulation(packed)
        img = lg.Image(ctx, 36, 2111, BOUNDS)
        for _ in range(3):
            for name, pieces in (("default", {}), ("small", dict(min_piece=2048, max_piece=8192))):
                ctx.set_tuning(**dict(before, **tuning, **pieces))
                img.clear()
                img.accumulate(segs)
                images[name] = img.accum()
                for _ in range(3):
                    t = time.perf_counter()
                    img.accumulate(segs)
                    best[name] = min(best.get(name, 1.0), time.perf_counter() - t)
    finally:
        ctx.set_packed_accumulation(True)
        ctx.set_tuning(**before)
    np.testing.assert_array_equal(images["default"], images["small"])
    print("default pieces %.0f us, up to 8192 pairs %.0f us" % (1e6 * best["default"], 1e6 * best["small"]))
    assert best["default"] < 1.12 * best["small"]
