"""Rays from far outside the objects: culling by bounding boxes returns the segments of the pass over
every object, bit for bit (lg_tuning.bvh_min_objects changes no result), also where the FP32
coordinates of a ray's origin are coarser than the boxes' own padding. Small and thin objects, whose
boxes have edges everywhere, near and beyond the default threshold; trees of more than two primitives
beside them; origins at 60 to 30000 units (FP32 rays of scenes beyond 64 test every object)."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import configs
from light_garden_amd import geo as G
from test_gpu_bvh import NEVER
from test_gpu_cull import segments

pytestmark = pytest.mark.gpu


def confetti(n, trees):
    from test_gpu_trace import nested_logic_zoo
    rng = np.random.default_rng(n)
    objs = list(nested_logic_zoo().objects) if trees else []
    while len(objs) < n:
        x, y = (float(v) for v in rng.uniform(-0.9, 0.9, 2))
        s = float(rng.uniform(0.01, 0.05))
        kind = len(objs) % 4
        if kind == 0:
            objs.append(lg.Object(G.Rect((x, y), G.rotation(float(rng.uniform(0, 3.1))), s, 2 * s), lg.Material(1.4)))
        elif kind == 1:
            objs.append(lg.Object.new_mirror((x, y), (x + s, y)))
        elif kind == 2:
            objs.append(lg.Object.new_mirror((x, y), (x, y + s)))
        else:
            objs.append(lg.Object(lg.Circle((x, y), s), lg.Material(1.5)))
    return objs


@pytest.mark.parametrize("fp64", [False, True], ids=["fp32", "fp64"])
@pytest.mark.parametrize("reach", [60.0, 300.0, 30000.0])
@pytest.mark.parametrize("n,trees", [(9, False), (70, False), (70, True)])
def test_far_origins(ctx, n, trees, reach, fp64):
    lights = []
    for a in (0.3, 0.8, 2.2, 3.9):
        o, d = np.array([np.cos(a), np.sin(a)]) * reach, np.array([-np.sin(a), np.cos(a)]) * 1.2
        for s in (-1, 1):  # one of the two faces the objects
            lights.append(lg.DirectionalLight([1.0, 1.0, 1.0, 1.0], 10000, G.LineSegment(tuple(o + s * d), tuple(o - s * d))))
    scene = configs.Scene(confetti(n, trees), lights, max_bounce=3, cutoff=(0.001,) * 4)
    before = ctx.tuning()
    try:
        full = segments(ctx, scene, fp64, NEVER)
        boxes = segments(ctx, scene, fp64, 1)
    finally:
        ctx.set_tuning(**before)
    assert np.bincount((full[0] >> np.uint64(24)).astype(int)).max() > 1
    for a, b in zip(full, boxes):
        np.testing.assert_array_equal(a, b)
