"""Batched frames of 64, 65 and 130 uneven scenes, scenes without segments among them: up to 64 scenes
every workgroup of the count pass makes the bin layout, beyond that a kernel of its own does. Each image
equals, bit for bit, the scene rendered alone."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import configs

pytestmark = pytest.mark.gpu


def small_scenes(n):
    rng = configs.SplitMix64(n)
    out = []
    for i in range(n):
        objs = configs.random_objects(rng, rng.randint(0, 12), first_type=i % 4)
        rays = 40000 if i == 7 else rng.randint(1, 700)
        lights = configs.random_lights(rng, [rays], [i % 3])
        sc = configs.Scene(objs, lights, max_bounce=rng.randint(1, 5), width=[64, 130, 257][i % 3], height=[64, 200][i % 2])
        if i % 13 == 5 or i == n - 1:
            sc.max_bounce = 0  # no segments
        out.append(sc)
    return out


def tracer(ctx, sc):
    tr = lg.Tracer(ctx, sc.canvas)
    for o in sc.objects:
        tr.push_object(o)
    for l in sc.lights:
        tr.push_light(l)
    tr.max_bounce = sc.max_bounce
    tr.cutoff_color = list(sc.cutoff)
    return tr


@pytest.mark.parametrize("n", [64, 65, 130])
def test_images_equal_scenes_alone(ctx, n):
    scenes = small_scenes(n)
    trs = [tracer(ctx, s) for s in scenes]
    segs = [lg.Segments(ctx) for _ in scenes]
    imgs = [lg.Image(ctx, s.width, s.height, s.canvas) for s in scenes]
    own, alone = lg.Segments(ctx), {}
    for k, (tr, s) in enumerate(zip(trs, scenes)):
        img = lg.Image(ctx, s.width, s.height, s.canvas)
        tr.render(own, img)
        alone[k] = (own.count(), img.accum(), img.rgba16f())
        img.close()
    assert min(c for c, _, _ in alone.values()) == 0
    for _ in range(2):  # the second frame replays the first's launches
        lg.batch_render(ctx, trs, segs, imgs)
        for k in range(n):
            assert segs[k].count() == alone[k][0]
            np.testing.assert_array_equal(imgs[k].accum(), alone[k][1])
            np.testing.assert_array_equal(imgs[k].rgba16f(), alone[k][2])
    for x in trs + segs + imgs + [own]:
        x.close()
