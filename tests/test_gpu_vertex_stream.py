"""The sample-stream walk with a colour per vertex (default blend, two-channel frames, 64-pixel tiles,
1024-thread workgroups) at its edge cases: streams that are whole multiples of 64 samples, 64
records in one step, waves that mix lengths, and waves that mix two colours with one. Each image equals the
per-pair walk's (512-thread workgroups take it) bit for bit, and the FP64 accumulation of the same
segments within the bound that the walk with one colour per segment keeps (the FP32 interpolation
adds some 1e-7); a frame with another blend takes the per-pair walk at either size."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import abi
from test_gpu_streams import full_crossings, mixed_lengths, one_sample

pytestmark = pytest.mark.gpu

KINDS = {"full_crossings": full_crossings, "one_sample": one_sample, "mixed_lengths": mixed_lengths}


def accumulate(ctx, pos, c0, c1, side, tile_block, blend=None):
    before = ctx.tuning()
    try:
        ctx.set_tuning(tile=64, tile_block=tile_block)
        segs = lg.Segments(ctx, capacity=len(pos), vertex_colors=True)
        segs.upload(pos, c0, c1)
        img = lg.Image(ctx, side, side, (-1.0, 1.0, -1.0, 1.0))
        if blend is not None:
            img.set_blend(color=blend)
        img.accumulate(segs)
        return img.accum()
    finally:
        ctx.set_tuning(**before)


@pytest.mark.parametrize("kind", list(KINDS))
def test_vertex_stream_equals_pair_walk_and_oracle(ctx, orc, kind):
    rng = np.random.default_rng(51 + list(KINDS).index(kind))
    side, n = 512, 6000
    pos = KINDS[kind](rng, side, n).astype(np.float32).astype(np.float64)
    c0 = rng.uniform(0.0, 0.01, (n, 4)).astype(np.float32)
    c1 = rng.uniform(0.0, 0.01, (n, 4)).astype(np.float32)
    c1[::3] = c0[::3]
    stream = accumulate(ctx, pos, c0, c1, side, 1024)
    pairs = accumulate(ctx, pos, c0, c1, side, 512)
    assert np.array_equal(stream, pairs)
    ref = orc.accumulate_f64(pos, c0, c1, abi.LgView(-1.0, 1.0, -1.0, 1.0, side, side), threads=8)
    e = orc.rel_l1(stream, ref)
    print("%s: rel L1 %.3e, accumulated %.6g" % (kind, e, stream[..., 0].sum()))
    assert stream[..., 0].sum() > 0
    assert e < 1e-5


def test_other_blends_take_the_pair_walk(ctx):
    rng = np.random.default_rng(57)
    side, n = 512, 3000
    pos = mixed_lengths(rng, side, n)
    c0, c1 = (rng.uniform(0.0, 0.1, (n, 4)).astype(np.float32) for _ in range(2))
    blend = (abi.BF_SRC_ALPHA, abi.BF_ONE, abi.BO_ADD)
    a, b = (accumulate(ctx, pos, c0, c1, side, block, blend) for block in (1024, 512))
    assert a[..., 0].sum() > 0
    assert np.array_equal(a, b)
    assert not np.array_equal(a, accumulate(ctx, pos, c0, c1, side, 1024))
