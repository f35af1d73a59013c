"""Trace items of a frame of several scenes: the frame's own sizes give the bits of small items."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import configs

pytestmark = pytest.mark.gpu


def frame(scenes, **tuning):
    ctx = lg.Context(0)
    ctx.set_tuning(**tuning)
    trs = []
    for sc in scenes:
        tr = lg.Tracer(ctx, sc.canvas)
        for o in sc.objects:
            tr.push_object(o)
        for l in sc.lights:
            tr.push_light(l)
        tr.max_bounce = 2
        trs.append(tr)
    segs = [lg.Segments(ctx) for _ in scenes]
    imgs = [lg.Image(ctx, 256, 256, sc.canvas) for sc in scenes]
    lg.batch_render(ctx, trs, segs, imgs)
    return [(np.sort(s.download()[3]), i.accum().copy()) for s, i in zip(segs, imgs)]


# 2048 workgroups (eight to each of 256 compute units, two scenes): a share of 256 rays and just
# above, of 512 and just above (items of 512), just above 1024 (items of half a share)
@pytest.mark.parametrize("total", [256 * 2048, 256 * 2048 + 1, 512 * 2048, 512 * 2048 + 1, 1024 * 2048 + 77])
def test_frame_items_equal_small_items(total):
    few = 30007
    scenes = [configs.large_single(num_rays=total - few, seed=2, width=256),
              configs.large_single(num_rays=few, seed=5, width=256)]
    own = frame(scenes, rays_per_item=4096)
    small = frame(scenes, rays_per_item=256)
    for (ka, ia), (kb, ib) in zip(own, small):
        assert np.array_equal(ka, kb)
        assert np.array_equal(ia, ib)
