"""Culling by bounding boxes returns the same segments, bit for bit, as the pass over every object
(reference: tracer.rs:413-423), at the sizes where its lists can go wrong: one object, a last block of
one and of four objects, full blocks, several blocks, every kind of object in one block, trees of
more than two primitives beside them (which the blocks do not hold), axis-parallel rays, and FP64
rays from far outside the objects (whose rounding to FP32 is wider than the boxes' padding)."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import configs
from light_garden_amd import geo as G
from test_gpu_bvh import NEVER

pytestmark = pytest.mark.gpu


def field(n, trees):
    from test_gpu_trace import nested_logic_zoo, shape_zoo
    zoo = list(shape_zoo().objects) + (list(nested_logic_zoo().objects) if trees else [])
    rng = np.random.default_rng(n)
    objs = zoo[:n]
    while len(objs) < n:
        x, y = rng.uniform(-2.0, 2.0, 2)
        objs.append(lg.Object(lg.Circle((float(x), float(y)), float(rng.uniform(0.02, 0.1))), lg.Material(1.5)))
    lights = [lg.PointLight((0.03, -0.41), 700, [1.0, 0.9, 0.8, 1.0]),
              lg.DirectionalLight([0.5, 0.6, 1.0, 1.0], 500, G.LineSegment((-1.5, -2.5), (1.5, -2.5))),
              lg.DirectionalLight([0.5, 0.6, 1.0, 1.0], 300, G.LineSegment((-2.5, 1.25), (-2.5, -1.0)))]
    return configs.Scene(objs, lights, max_bounce=6, cutoff=(0.001, 0.001, 0.001, 0.001))


def segments(ctx, scene, fp64, min_objects):
    ctx.set_tuning(bvh_min_objects=min_objects)
    tr = lg.Tracer(ctx, scene.canvas)
    for o in scene.objects:
        tr.push_object(o)
    for l in scene.lights:
        tr.push_light(l)
    tr.max_bounce = scene.max_bounce
    tr.cutoff_color = list(scene.cutoff)
    tr.fp64 = fp64
    segs = tr.trace()
    pos, c0, c1, key = segs.download()
    if fp64:
        pos = segs.download_pos64()
    segs.close()
    tr.close()
    o = np.argsort(key, kind="stable")
    return key[o], pos[o], c0[o], c1[o]


@pytest.mark.parametrize("far", [False, True], ids=["near", "far"])
@pytest.mark.parametrize("fp64", [False, True], ids=["fp32", "fp64"])
@pytest.mark.parametrize("n,trees", [(1, False), (4, False), (64, False), (65, False), (68, True), (200, True)])
def test_boxes_equal_full_walk(ctx, n, trees, fp64, far):
    if far and not fp64:
        pytest.skip("FP32 rays carry no more precision than the boxes")
    scene = field(n, trees)
    if far:
        for s in (-1.5, 1.5):  # one of the two faces the objects
            line = G.LineSegment((30000.0 - 2 * s, 20000.0 + 3 * s), (30000.0 + 2 * s, 20000.0 - 3 * s))
            scene.lights.append(lg.DirectionalLight([1.0, 1.0, 1.0, 1.0], 400, line))
    before = ctx.tuning()
    try:
        full = segments(ctx, scene, fp64, NEVER)
        boxes = segments(ctx, scene, fp64, 1)
    finally:
        ctx.set_tuning(**before)
    assert len(full[0]) > 1400
    if far:
        assert np.bincount((full[0] >> np.uint64(24)).astype(int))[1500:].max() > 1
    for a, b in zip(full, boxes):
        np.testing.assert_array_equal(a, b)
