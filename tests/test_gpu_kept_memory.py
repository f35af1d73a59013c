"""Device memory that calls keep between them is bounded: after trace_all of a large scene the device
has all but the kept scratch's bound (64 MiB) back, after a StringMod of many points all of it, and
the calls give the same results as before."""
import numpy as np
import pytest
import torch

import light_garden_amd as lg
from light_garden_amd import configs, string_mod

pytestmark = pytest.mark.gpu

MIB = 1 << 20
KEPT = 64 * MIB
SLACK = 8 * MIB  # allocation granularity


def free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_trace_all_gives_its_memory_back(ctx):
    torch.zeros(1, device="cuda")
    n = 3_000_000
    scene = configs.Scene([], [lg.PointLight((0.1, 0.2), n, [0.01] * 4)], max_bounce=1)
    tr = lg.Tracer(ctx, scene.canvas)
    tr.push_light(scene.lights[0])
    tr.max_bounce = 1
    segs = tr.trace()  # the scene's own ray queues stay with it
    want = segs.download()[0]
    segs.close()
    before = free()
    xy, rgba = tr.trace_all()
    kept = before - free()
    print("trace_all of %d segments keeps %.1f MiB" % (len(xy) // 2, kept / MIB))
    assert len(xy) == 2 * n and kept <= KEPT + SLACK  # (120 MB of segments, 150 MB of scratch)
    assert np.abs(xy.reshape(-1, 4)[:, :2] - [0.1, 0.2]).max() < 1e-6 and len(want) == n
    again = tr.trace_all()
    np.testing.assert_array_equal(again[0], xy)
    np.testing.assert_array_equal(again[1], rgba)
    tr.close()


def test_string_mods_keep_no_points(ctx):
    torch.zeros(1, device="cuda")
    m = 6_000_000
    segs = lg.Segments(ctx, capacity=m, vertex_colors=True)
    small = [lg.StringMod(modulo=5000, num=2, scale=0.9, color=[0.01] * 4)]
    string_mod.draw(ctx, small, segs)
    want = segs.download()[0]
    before = free()
    assert string_mod.draw(ctx, [lg.StringMod(modulo=m, num=2, scale=0.9, color=[0.01] * 4)], segs) == m
    kept = before - free()
    print("a draw of %d points keeps %.1f MiB" % (m, kept / MIB))
    assert kept <= SLACK  # (the points: 92 MiB)
    string_mod.draw(ctx, small, segs)
    np.testing.assert_array_equal(segs.download()[0], want)
    segs.close()
