"""Ordered vertices of a segment buffer (lg_segments_download_vertices, the download behind
trace_all): equal, value for value, to the downloaded arrays sorted by key on the host. Sizes where
the device ordering can go wrong: no segment, one ray, a buffer of several copy chunks, rays with
more segments than the device ranks (ordered on the host), FP64 end points, and a buffer that was
not traced (with a colour per vertex)."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import configs

pytestmark = pytest.mark.gpu


def tracer(ctx, scene, fp64=False):
    tr = lg.Tracer(ctx, scene.canvas)
    for o in scene.objects:
        tr.push_object(o)
    for l in scene.lights:
        tr.push_light(l)
    tr.max_bounce = scene.max_bounce
    tr.cutoff_color = list(scene.cutoff)
    tr.fp64 = fp64
    return tr


def by_host(segs, fp64=False):
    pos, c0, c1, key = segs.download()
    if fp64:
        pos = segs.download_pos64()
    o = np.argsort(key, kind="stable")
    return pos[o].astype(np.float64).reshape(-1, 2), np.stack([c0[o], c1[o]], 1).reshape(-1, 4)


def nested_glass(n_rays):
    """Concentric circles of alternating index: most hits split, so a ray's tree doubles per bounce."""
    objs = [lg.Object(lg.Circle((0.0, 0.0), 0.9 - 0.05 * k), lg.Material(1.1 + 0.35 * (k % 2))) for k in range(12)]
    lights = [lg.PointLight((0.13, 0.07), n_rays, [1.0, 1.0, 1.0, 1.0])]
    return configs.Scene(objs, lights, max_bounce=14, cutoff=(0.0, 0.0, 0.0, 0.0))


@pytest.mark.parametrize("fp64", [False, True], ids=["fp32", "fp64"])
@pytest.mark.parametrize("scene", [configs.plain_small(1), configs.plain_small(257), configs.large_single(70000),
                                   nested_glass(5)], ids=["one_ray", "257_rays", "chunks", "long_rays"])
def test_vertices_equal_host_sort(ctx, scene, fp64):
    tr = tracer(ctx, scene, fp64)
    segs = tr.trace()
    want_xy, want_rgba = by_host(segs, fp64)
    xy, rgba = segs.vertices()
    np.testing.assert_array_equal(xy, want_xy)
    np.testing.assert_array_equal(rgba, want_rgba)
    for _ in range(2):  # trace_all's kept buffer, twice
        xy, rgba = tr.trace_all()
        np.testing.assert_array_equal(xy, want_xy)
        np.testing.assert_array_equal(rgba, want_rgba)
    n = segs.count()
    if scene.n_rays() == 70000:
        assert n > 2 * (1 << 17)
    if scene.n_rays() == 5:
        assert np.bincount((segs.download()[3] >> np.uint64(24)).astype(int)).max() > 2048


def test_vertices_of_other_buffers(ctx):
    rng = np.random.default_rng(3)
    pos = rng.uniform(-1, 1, (1000, 4))
    c0, c1 = rng.uniform(0, 1, (2, 1000, 4)).astype(np.float32)
    segs = lg.Segments(ctx, vertex_colors=True)
    assert segs.vertices()[0].shape == (0, 2)
    segs.upload(pos, c0, c1)
    xy, rgba = segs.vertices()
    np.testing.assert_array_equal(xy, pos.astype(np.float32).astype(np.float64).reshape(-1, 2))
    np.testing.assert_array_equal(rgba, np.stack([c0, c1], 1).reshape(-1, 4))
    # traced, then uploaded over: the rays are forgotten
    scene = configs.plain_small(300)
    tr = tracer(ctx, scene)
    tr.trace(segs)
    want = by_host(segs)
    got = segs.vertices()
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])
    segs.upload(pos, c0, c1)
    np.testing.assert_array_equal(segs.vertices()[1], np.stack([c0, c1], 1).reshape(-1, 4))
