"""Ordered vertices where the device has no room for the ordering's scratch (the rest of its memory is held
elsewhere): the host orders the buffer, with the same values, and later calls are as before."""
import numpy as np
import pytest
import torch

import light_garden_amd as lg
from light_garden_amd import configs

pytestmark = pytest.mark.gpu


def test_host_orders_without_device_scratch(ctx):
    n = 24_000_000  # 40 bytes of scratch each, 8 per ray: 1.1 GB
    scene = configs.Scene([], [lg.PointLight((0.1, 0.2), n, [0.01] * 4)], max_bounce=1)
    tr = lg.Tracer(ctx, scene.canvas)
    tr.push_light(scene.lights[0])
    tr.max_bounce = 1
    segs = tr.trace()
    assert segs.count() == n
    torch.zeros(1, device="cuda")
    held = torch.empty(torch.cuda.mem_get_info()[0] - (256 << 20), dtype=torch.uint8, device="cuda")
    print("%d MiB free" % (torch.cuda.mem_get_info()[0] >> 20))
    try:
        xy, rgba = segs.vertices()
    finally:
        del held
        torch.cuda.empty_cache()
    again = segs.vertices()  # on the device
    np.testing.assert_array_equal(xy, again[0])
    np.testing.assert_array_equal(rgba, again[1])
    small = lg.Segments(ctx)
    tr2 = lg.Tracer(ctx, scene.canvas)
    tr2.push_light(lg.PointLight((0.1, 0.2), 1000, [0.01] * 4))
    img = lg.Image(ctx, 64, 64, scene.canvas)
    tr2.render(small, img)
    assert small.count() == 1000 and img.accum().any()
    for x in (tr, tr2, segs, small, img):
        x.close()
