"""Levels of a deposit's weight where segments of one colour are summed as weights: with n pairs in a
tile (32768 at most count) a 32-bit word has room for floor((2^32 - 1) / n) levels, and a weight has them
all, as a channel value has in the walk by colours. Horizontal lines, each alone in its two rows of
a tile whose other pairs crowd one pixel: their deposits within half a level of the exact weights."""
import numpy as np
import pytest

import light_garden_amd as lg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("color", [0.99, 0.5, 0.0039])
@pytest.mark.parametrize("n", [20000, 32768, 70001])
def test_weights_keep_their_levels(ctx, n, color):
    rng = np.random.default_rng(n)
    rows = np.arange(2, 62, 2)
    f = rng.integers(1, 1 << 18, len(rows)) / float(1 << 18)  # exact in FP32 at these coordinates
    pos = np.empty((n, 4), np.float64)
    pos[:] = (40.0, 64.0 - 10.5, 41.0, 64.0 - 10.5)  # the crowd: column 40, row 10
    y = 64.0 - (rows + 0.5 + f)
    pos[:len(rows)] = np.stack([np.zeros(len(rows)), y, np.full(len(rows), 32.0), y], 1)
    assert (pos.astype(np.float32) == pos).all()
    col = np.full((n, 4), color, np.float32)
    segs = lg.Segments(ctx)
    segs.upload(pos, col)
    img = lg.Image(ctx, 64, 64, (0.0, 64.0, 0.0, 64.0))
    img.accumulate(segs)
    got = img.accum().astype(np.float64)[:, :32]
    levels = (2 ** 32 - 1) // min(n, 32768)
    c = col[0].astype(np.float64)
    c[3] *= c[3]
    worst = 0.0
    for r, w in zip(rows, f):
        for row, weight in ((r, 1.0 - w), (r + 1, w)):
            worst = max(worst, np.abs(got[row] / c - weight).max())
    print("n %d: error %.3e of a sample, half a level is %.3e" % (n, worst, 0.5 / levels))
    # half a level, the line's place in steps of 2^-22, FP32 sums and colours
    assert worst <= 0.5 / levels + 2.0 ** -22 + 2.0 ** -23
