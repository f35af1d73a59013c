"""Ordered vertices of rays with very many segments: up to 65536 of one ray are ranked on the device,
buffers with a longer ray are sorted on the host. Equal, value for value, to the downloaded arrays
sorted by key; and no slower than that sort, which trace_all was before it had an order of its own."""
import time

import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import configs
from test_gpu_order import by_host, nested_glass, tracer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp64", [False, True], ids=["fp32", "fp64"])
@pytest.mark.parametrize("rays,bounces,longest", [(3, 16, (60000, 65536)), (2, 17, (65537, 1 << 17)), (1, 18, (1 << 17, 1 << 18))])
def test_long_rays_equal_host_sort(ctx, rays, bounces, longest, fp64):
    scene = nested_glass(rays)
    scene.max_bounce = bounces
    tr = tracer(ctx, scene, fp64)
    segs = tr.trace()
    most = np.bincount((segs.download()[3] >> np.uint64(24)).astype(int)).max()
    assert longest[0] <= most <= longest[1]
    want = by_host(segs, fp64)
    got = segs.vertices()
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])
    segs.close()
    tr.close()


def test_no_slower_than_the_host_sort(ctx):
    scene = nested_glass(40)
    tr = tracer(ctx, scene)
    segs = tr.trace()

    def best(f):
        out = []
        for _ in range(7):
            t = time.perf_counter()
            f()
            out.append(time.perf_counter() - t)
        return min(out)

    def sorted_in_numpy():
        pos, col, _, key = segs.download()
        o = np.argsort(key, kind="stable")
        return np.asarray(pos, np.float64)[o].reshape(-1, 2), np.repeat(col[o], 2, axis=0)

    own, sort = best(segs.vertices), best(sorted_in_numpy)
    print("%d segments: %.2f ms, sorted in numpy %.2f ms" % (segs.count(), 1e3 * own, 1e3 * sort))
    assert own <= sort
