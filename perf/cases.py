"""Performance cases: the work that programs built on light_garden_amd have it do, through the
package's public entry points.

A case is a dict of plain values; `kind` says which entry points it takes:

  frame    one Tracer.render: trace, accumulate, resolve. With `edit`, an object is replaced
           before the frame, as an editor does on every mouse move of a drag
  batch    one batch_render of several uneven scenes
  trace    one Tracer.trace_all: the vertex pairs in emission order on the host (`fp64`: traced
           in FP64 end to end)
  strings  string_mod.draw of `mods` StringMods, then clear, accumulate, resolve (`colors`:
           modulo colours per StringMod; `nested`: drawn over the crossings of another's lines)
  lines    host segments uploaded, then clear, accumulate, resolve: the drop-in for a program
           that keeps its own tracer (`vertex_colors`: a colour per end point)
  serve    a burst of render requests through a Server, some of them with an edit

Scenes, colours and sizes follow this repository's workloads (light_garden_amd/configs.py: the
plain small scene, the large single scene, the batched uneven scenes, the string-mod picture;
tests/golden/default.ron: the scene the editor starts with). Each state holds a Context of its
own, as a program holds one, at the library's default settings.
"""
import math
import random

import numpy as np
import torch

import light_garden_amd as lg
from light_garden_amd import abi, string_mod

BOUNDS = (-1.0, 1.0, -1.0, 1.0)
T_MIN = 1e-5


# ---- the cases ------------------------------------------------------------------------------------
def listed():
    return [
        # the first light a user drops into an empty editor, dragged about: the smallest frame
        dict(name="edit_tiny", kind="frame", scene="mixed", rays=360, objects=2, bounces=5, width=640, height=480,
             edit=True),
        # the editor's start-up scene (a point and a spot light, three objects) while one is dragged
        dict(name="edit_default", kind="frame", scene="default", rays=12000, objects=3, bounces=5, width=1280,
             height=720, edit=True),
        # the plain small scene of the benchmark, rendered again and again
        dict(name="frame_small", kind="frame", scene="small", rays=20000, objects=4, bounces=5, width=1024,
             height=1024, edit=False),
        # an odd window, an uneven number of rays, every kind of object
        dict(name="frame_odd", kind="frame", scene="all", rays=75011, objects=23, bounces=8, width=1366, height=769,
             edit=False),
        # the benchmark's large single scene
        dict(name="frame_large", kind="frame", scene="mixed", rays=1000000, objects=64, bounces=10, width=2048,
             height=2048, edit=False),
        # a sheet of uneven scenes in one call
        dict(name="batch_uneven", kind="batch", scenes=20, rays=800000, objects=160, side=1536),
        # trace_all of the plain small scene: the vertices on the host, in order
        dict(name="trace_small", kind="trace", scene="small", rays=20000, objects=4, bounces=5, fp64=False),
        # the FP64 option, on a scene with every kind of object
        dict(name="trace_fp64", kind="trace", scene="all", rays=40009, objects=12, bounces=6, fp64=True),
        # the benchmark's string-mod picture
        dict(name="strings_large", kind="strings", points=100000, mods=16, colors=0, nested=False, width=4096,
             height=4096),
        # string art with modulo colours: a colour of its own at each end of a line
        dict(name="strings_colored", kind="strings", points=20011, mods=3, colors=4, nested=False, width=2048,
             height=1536),
        # another program's segments, uploaded and drawn
        dict(name="lines_upload", kind="lines", segments=100003, vertex_colors=False, width=1920, height=1080),
        # a render server under a burst of requests, every third one with an edit
        dict(name="serve_burst", kind="serve", requests=24, rays=60000, objects=24, side=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["edit", "frame", "frame", "batch", "trace", "trace", "strings", "colored", "nested", "lines",
                       "serve"])
    if kind in ("edit", "frame"):
        edit = kind == "edit"
        return dict(kind="frame", scene=rng.choice(["small", "mixed", "all", "default"]),
                    rays=_log(rng, 300, 20000 if edit else 600000), objects=_log(rng, 1, 64),
                    bounces=rng.randint(3, 10), width=_log(rng, 500, 2048), height=_log(rng, 400, 1600), edit=edit)
    if kind == "batch":
        return dict(kind="batch", scenes=rng.randint(3, 20), rays=_log(rng, 5000, 600000), objects=_log(rng, 4, 160),
                    side=_log(rng, 500, 1536))
    if kind == "trace":
        fp64 = rng.random() < 0.4
        return dict(kind="trace", scene=rng.choice(["small", "mixed", "all", "default"]), rays=_log(rng, 300, 100000),
                    objects=_log(rng, 1, 48), bounces=rng.randint(3, 8), fp64=fp64)
    if kind == "strings":
        return dict(kind="strings", points=_log(rng, 300, 100000), mods=rng.randint(1, 12), colors=0, nested=False,
                    width=_log(rng, 700, 4096), height=_log(rng, 700, 4096))
    if kind == "colored":
        return dict(kind="strings", points=_log(rng, 300, 30000), mods=rng.randint(1, 4), colors=rng.randint(1, 6),
                    nested=False, width=_log(rng, 700, 2500), height=_log(rng, 700, 2000))
    if kind == "nested":
        return dict(kind="strings", points=_log(rng, 100, 1500), mods=1, colors=rng.choice([0, 3]), nested=True,
                    width=_log(rng, 700, 2048), height=_log(rng, 700, 2048))
    if kind == "lines":
        return dict(kind="lines", segments=_log(rng, 500, 300000), vertex_colors=rng.random() < 0.3,
                    width=_log(rng, 500, 3840), height=_log(rng, 400, 2160))
    return dict(kind="serve", requests=rng.randint(4, 32), rays=_log(rng, 2000, 60000), objects=_log(rng, 2, 48),
                side=_log(rng, 400, 1024))


# ---- scenes, as plain values ------------------------------------------------------------------------
# An object is (shape, parameters, refractive index or None for a mirror); a light (kind, position,
# direction or band end, rays, colour).
def _hue(rng, level):
    u = [rng.uniform(0.05, 1.0) for _ in range(3)]
    m = max(u)
    return [float(np.float32(level * v / m)) for v in u] + [float(np.float32(level))]


def _objects(rng, n, shapes):
    out = []
    for i in range(n):
        s = shapes[i % len(shapes)]
        cx, cy, a = rng.uniform(-0.9, 0.9), rng.uniform(-0.9, 0.9), rng.uniform(0.0, math.pi)
        ior = rng.uniform(1.3, 1.8)
        if s == "circle":
            out.append((s, (cx, cy, rng.uniform(0.02, 0.15)), ior))
        elif s == "rect":
            out.append((s, (cx, cy, a, rng.uniform(0.02, 0.2), rng.uniform(0.02, 0.2)), ior))
        elif s == "ellipse":
            out.append((s, (cx, cy, a, rng.uniform(0.03, 0.15), rng.uniform(0.02, 0.1)), ior))
        elif s == "lens":
            r = rng.uniform(0.03, 0.15)
            out.append((s, (cx, cy, a, r, rng.uniform(0.5, 1.6) * r), ior))
        elif s == "poly":
            r, k = rng.uniform(0.04, 0.15), rng.randint(3, 7)
            out.append((s, (cx, cy, a, tuple((r * math.cos(2 * math.pi * j / k), r * math.sin(2 * math.pi * j / k))
                                             for j in range(k))), ior))
        elif s == "mirror":
            h = 0.5 * rng.uniform(0.05, 0.3)
            out.append((s, (cx - h * math.cos(a), cy - h * math.sin(a), cx + h * math.cos(a), cy + h * math.sin(a)),
                        None))
        else:  # curved mirror: a shallow cubic over a chord
            h = 0.5 * rng.uniform(0.1, 0.4)
            ux, uy = math.cos(a), math.sin(a)
            b = rng.uniform(-0.5, 0.5) * h
            out.append(("curve", (cx - h * ux, cy - h * uy, cx - 0.4 * h * ux - b * uy, cy - 0.4 * h * uy + b * ux,
                                  cx + 0.4 * h * ux - b * uy, cy + 0.4 * h * uy + b * ux, cx + h * ux, cy + h * uy),
                        None))
    return out


def _lights(rng, rays, kinds, level):
    base = rays // len(kinds)
    out = []
    for i, k in enumerate(kinds):
        n = rays - base * (len(kinds) - 1) if i == 0 else base
        px, py, a = rng.uniform(-0.9, 0.9), rng.uniform(-0.9, 0.9), rng.uniform(0.0, 2 * math.pi)
        if k == "band":
            ex, ey = 0.2 * math.cos(a), 0.2 * math.sin(a)
            out.append((k, (px - ex, py - ey), (px + ex, py + ey), n, _hue(rng, level)))
        else:
            out.append((k, (px, py), (math.cos(a), math.sin(a)), n, _hue(rng, level)))
    return out


def _scene(kind, rays, objects, rng):
    if kind == "small":  # the plain small scene, shifted a little by the seed; more objects follow the four
        j = [rng.uniform(-0.03, 0.03) for _ in range(6)]
        objs = [("circle", (0.5 + j[0], j[1], 0.2), 1.5), ("rect", (-0.5 + j[2], 0.3 + j[3], 0.0, 0.3, 0.2), 1.33),
                ("mirror", (-0.6, -0.6 + j[4], 0.6, -0.5 + j[4]), None),
                ("curve", (0.6928, -0.2 + j[5], 0.8359, 0.0479 + j[5], 0.8359, 0.3521 + j[5], 0.6928, 0.6 + j[5]), None)]
        objs = objs[:objects] + _objects(rng, max(0, objects - 4), ["circle", "rect", "lens", "mirror"])
        return objs, [("point", (0.0, 0.0), (1.0, 0.0), rays, [float(np.float32(0.01))] * 4)]
    if kind == "default":  # the editor's start-up scene: a wide lens, a curved mirror, a rect around the light
        dx = rng.uniform(-0.05, 0.05)
        objs = [("lens", (-0.0228 + dx, -0.1, -0.5 * math.pi, 2.0, 3.8), 1.05),
                ("curve", (-0.6228, 0.4, -0.3228, 0.8, 0.2772, 0.8, 0.5772, 0.4), None),
                ("rect", (-0.0228 + dx, -0.5, 0.0, 0.4, 0.4), 1.73)]
        objs = objs[:objects] + _objects(rng, max(0, objects - 3), ["circle", "rect", "lens", "mirror"])
        spot = rays // 6
        return objs, [("point", (-0.0228 + dx, -0.5), (1.0, 0.0), rays - spot, _hue(rng, 0.0117)),
                      ("spot10", (0.95, -0.1), (-0.99999, 0.00394), spot, _hue(rng, 0.035))]
    shapes = ["circle", "rect", "lens", "mirror"] + (["curve", "ellipse", "poly"] if kind == "all" else [])
    objs = _objects(rng, objects, shapes)
    return objs, _lights(rng, rays, ["point", "spot", "band"] if rays >= 3000 else ["point"], 0.002)


def _aspect(width, height):
    a = width / height
    return (-a, a, -1.0, 1.0)


def _moved(obj, dx=0.013, dy=-0.007):
    """The object at another place; by default the dragged object's in the edited frame."""
    s, p, ior = obj
    if s in ("mirror", "curve"):
        return s, tuple(v + (dx if i % 2 == 0 else dy) for i, v in enumerate(p)), ior
    return s, (p[0] + dx, p[1] + dy) + tuple(p[2:]), ior


def _trace_scene(case, seed):
    """(scene, canvas) of a trace: the case fixes the arrangement (so that every seed gives as many
    segments), the seed pans it, canvas and all, and colours its lights."""
    rng = random.Random(seed)
    objs, lights = _scene(case["scene"], case["rays"], case["objects"], random.Random(case["rays"] + case["objects"]))
    dx, dy = rng.uniform(-0.2, 0.2), rng.uniform(-0.2, 0.2)
    lights = [(k, (p[0] + dx, p[1] + dy), (q[0] + dx, q[1] + dy) if k == "band" else q, n, _hue(rng, c[3]))
              for k, p, q, n, c in lights]
    return ([_moved(o, dx, dy) for o in objs], lights), (BOUNDS[0] + dx, BOUNDS[1] + dx, BOUNDS[2] + dy, BOUNDS[3] + dy)


# the sizes of a batch or burst come from the case, its scenes from the seed
def _batch_scenes(case, seed):
    size, rng = random.Random(case["rays"]), random.Random(seed)
    got = []
    for i in range(case["scenes"]):
        rays = max(3, _log(size, 1000, max(1001, case["rays"])))
        objects = _log(size, 1, max(2, case["objects"]))
        side = size.choice([case["side"], case["side"] // 2 + 1, case["side"] // 3])
        got.append((_scene("mixed", rays, objects, rng), size.randint(3, 12), side))
    return got


def _serve_scenes(case, seed):
    size, rng = random.Random(case["rays"]), random.Random(seed)
    got = []
    for i in range(case["requests"]):
        rays = max(3, _log(size, 1000, max(1001, case["rays"])))
        objects = size.randint(2, max(2, case["objects"]))
        side = size.choice([case["side"], case["side"] // 2 + 1])
        got.append((_scene("mixed", rays, objects, rng), size.randint(3, 8), side))
    return got


# ---- package objects ---------------------------------------------------------------------------------
def _lg_object(obj):
    s, p, ior = obj
    if s == "mirror":
        return lg.Object.new_mirror(p[:2], p[2:])
    if s == "curve":
        return lg.Object.new_curved_mirror(lg.CubicBezier([(p[i], p[i + 1]) for i in range(0, 8, 2)]))
    if s == "circle":
        g = lg.Circle((p[0], p[1]), p[2])
    elif s == "rect":
        g = lg.Rect((p[0], p[1]), lg.rotation(p[2]), p[3], p[4])
    elif s == "ellipse":
        g = lg.Ellipse((p[0], p[1]), p[3], p[4], lg.rotation(p[2]))
    elif s == "lens":
        g = lg.lens((p[0], p[1]), p[3], p[4])
        g.rotation = lg.rotation(p[2])
    else:
        g = lg.ConvexPolygon(p[3], (p[0], p[1]), lg.rotation(p[2]))
    return lg.Object(g, lg.Material(ior))


def _spot_angle(kind):
    return math.radians(10.0) if kind == "spot10" else math.pi / 6.0


def _lg_light(light):
    kind, pos, direction, n, color = light
    if kind == "point":
        return lg.PointLight(pos, n, color)
    if kind == "band":
        return lg.DirectionalLight(color, n, lg.LineSegment(pos, direction))
    return lg.SpotLight(pos, _spot_angle(kind), direction, n, color)


def _tracer(ctx, scene, bounces, canvas):
    t = lg.Tracer(ctx, canvas)
    t.max_bounce = bounces
    for o in scene[0]:
        t.push_object(_lg_object(o))
    for l in scene[1]:
        t.push_light(_lg_light(l))
    return t


class _Device:
    """A device buffer of the library for torch, without a copy (lg_image_device_ptrs)."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 2}


def _image(ctx, width, height, bounds):
    import ctypes as C
    img = lg.Image(ctx, width, height, bounds)
    a, h = C.c_void_p(), C.c_void_p()
    abi.call("lg_image_device_ptrs", img.handle, C.byref(a), C.byref(h))
    out = {"accum": torch.as_tensor(_Device(a.value, (height, width, 4), "<f4"), device="cuda"),
           "image": torch.as_tensor(_Device(h.value, (height, width, 4), "<f2"), device="cuda")}
    for view in out.values():
        view.owner = img  # the buffers live as long as the image: a view keeps it (and its context)
    return img, out


def _strings(case, seed):
    """The StringMods as plain dicts (points, num, color, modulo colours)."""
    rng = random.Random(seed)
    got = []
    for i in range(case["mods"]):
        cols = [(rng.randint(2, 9), rng.randint(0, 1), _hue(rng, 0.002)) for _ in range(case["colors"])]
        got.append(dict(modulo=case["points"], num=2 + i + rng.randint(0, 40), color=_hue(rng, 0.002), cols=cols))
    return got


def _lines(case, seed):
    r = np.random.RandomState(seed % (1 << 32))
    n = case["segments"]
    b = _aspect(case["width"], case["height"])
    p = r.uniform(-1.0, 1.0, (n, 2)) * [b[1], 1.0]
    a, l = r.uniform(0.0, 2 * np.pi, n), np.exp(r.uniform(np.log(0.02), np.log(1.5), n))
    q = p + np.stack([np.cos(a), np.sin(a)], 1) * l[:, None]
    pos = np.concatenate([p, q], 1).astype(np.float32)
    c0 = r.uniform(0.0005, 0.01, (n, 4)).astype(np.float32)
    c1 = r.uniform(0.0005, 0.01, (n, 4)).astype(np.float32) if case["vertex_colors"] else None
    return pos, c0, c1, b


def prepare(case, seed):
    ctx = lg.Context(0)
    s = {"case": case, "ctx": ctx}
    kind = case["kind"]
    if kind == "frame":
        scene = _scene(case["scene"], case["rays"], case["objects"], random.Random(seed))
        b = _aspect(case["width"], case["height"])
        s["tracer"] = _tracer(ctx, scene, case["bounces"], b)
        s["segs"] = lg.Segments(ctx)
        s["img"], s["out"] = _image(ctx, case["width"], case["height"], b)
        if case["edit"]:
            s["edit"] = _lg_object(_moved(scene[0][0]))
    elif kind == "batch":
        s["tracers"], s["segs"], s["imgs"], s["out"] = [], [], [], []
        for scene, bounces, side in _batch_scenes(case, seed):
            s["tracers"].append(_tracer(ctx, scene, bounces, BOUNDS))
            s["segs"].append(lg.Segments(ctx))
            img, out = _image(ctx, side, side, BOUNDS)
            s["imgs"].append(img)
            s["out"].append(out)
    elif kind == "trace":
        scene, canvas = _trace_scene(case, seed)
        s["tracer"] = _tracer(ctx, scene, case["bounces"], canvas)
        s["tracer"].fp64 = case["fp64"]
    elif kind == "strings":
        mods = [lg.StringMod(modulo=m["modulo"], num=m["num"], color=m["color"], scale=0.9,
                             modulo_colors=[lg.ModRemColor(*c) for c in m["cols"]]) for m in _strings(case, seed)]
        if case["nested"]:  # drawn over the crossings of 61 lines
            mods = [lg.StringMod(modulo=61, num=m.num, scale=0.9, color=m.color, nested=m) for m in mods]
        s["mods"] = mods
        s["segs"] = lg.Segments(ctx, vertex_colors=True)
        b = _aspect(case["width"], case["height"])
        s["img"], s["out"] = _image(ctx, case["width"], case["height"], b)
    elif kind == "lines":
        s["pos"], s["c0"], s["c1"], b = _lines(case, seed)
        s["segs"] = lg.Segments(ctx, vertex_colors=case["vertex_colors"])
        s["img"], s["out"] = _image(ctx, case["width"], case["height"], b)
    else:
        s["server"] = lg.Server(ctx)
        s["tracers"], s["imgs"], s["out"], s["edits"] = [], [], [], []
        for i, (scene, bounces, side) in enumerate(_serve_scenes(case, seed)):
            s["tracers"].append(_tracer(ctx, scene, bounces, BOUNDS))
            s["edits"].append((0, _lg_object(_moved(scene[0][0]))) if i % 3 == 0 else None)
            img, out = _image(ctx, side, side, BOUNDS)
            s["imgs"].append(img)
            s["out"].append(out)
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "frame":
        if "edit" in s:
            s["tracer"].replace_object(0, s["edit"])
        s["tracer"].render(s["segs"], s["img"])
        return s["out"]
    if kind == "batch":
        lg.batch_render(s["ctx"], s["tracers"], s["segs"], s["imgs"])
        return s["out"]
    if kind == "trace":
        xy, rgba = s["tracer"].trace_all()
        return {"xy": xy, "rgba": rgba}
    if kind == "strings":
        string_mod.draw(s["ctx"], s["mods"], s["segs"])
        s["img"].clear()
        s["img"].accumulate(s["segs"])
        s["img"].resolve()
        return s["out"]
    if kind == "lines":
        s["segs"].upload(s["pos"], s["c0"], s["c1"])
        s["img"].clear()
        s["img"].accumulate(s["segs"])
        s["img"].resolve()
        return s["out"]
    tickets = [s["server"].submit(t, i, edit=e) for t, i, e in zip(s["tracers"], s["imgs"], s["edits"])]
    for t in tickets:
        s["server"].wait(t)
    return s["out"]


# ---- what a pass cannot do without --------------------------------------------------------------------
def _trace_work(rays, objects, bounces):
    """(segments, flops) of a trace, from the ratios the benchmark's scenes show: about 1 + 0.35
    segments per ray and bounce, an interior test of about 30 flops per object and segment."""
    segs = rays * min(1.0 + 0.35 * bounces, 6.0)
    return segs, segs * (30.0 * objects + 52.0)


def _draw_work(segs, mean_px, width, height, seg_bytes=40):
    """(bytes, flops) of drawing: segments in, accumulator and RGBA16F out; a sample is two deposits
    of four channels."""
    return segs * seg_bytes + width * height * 24.0, segs * mean_px * 20.0


def work(case):
    kind = case["kind"]

    def frame(rays, objects, bounces, width, height):
        segs, ft = _trace_work(rays, objects, bounces)
        b, fd = _draw_work(segs, 0.3 * max(width, height) / (1.0 + 0.03 * objects), width, height)
        return segs * 40.0 + b, ft + fd

    if kind == "frame":
        b, f = frame(case["rays"], case["objects"], case["bounces"], case["width"], case["height"])
    elif kind in ("batch", "serve"):
        b = f = 0.0
        for scene, bounces, side in (_batch_scenes if kind == "batch" else _serve_scenes)(case, 1):
            x, y = frame(sum(l[3] for l in scene[1]), len(scene[0]), bounces, side, side)
            b, f = b + x, f + y
    elif kind == "trace":
        segs, f = _trace_work(case["rays"], case["objects"], case["bounces"])
        b = segs * 64.0  # two vertices of two doubles and four floats
    elif kind == "strings":
        segs = case["points"] * case["mods"]
        b, f = _draw_work(segs, 0.5 * case["height"], case["width"], case["height"], 96 if case["colors"] else 72)
    else:
        segs = case["segments"]
        b, f = _draw_work(segs, 0.15 * case["height"], case["width"], case["height"], 48 if case["vertex_colors"] else 32)
    return {"bytes": float(b), "flops": float(f)}


# ---- the same results in 64 bits, in plain torch ---------------------------------------------------
MOST_SAMPLES = 150_000_000  # more than this takes a plain scatter over a quarter of a minute


def _t(v):
    return torch.tensor(v, dtype=torch.float64, device="cuda")


def _dot(a, b):
    return a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1]


def _unit(v):
    return v / torch.sqrt(_dot(v, v))[..., None]


def _circle(o, d, c, r):
    """Chord of a circle: (meets, t in, t out, outward normals at both)."""
    l = o - c
    b, cc = _dot(l, d), _dot(l, l) - r * r
    disc = b * b - cc
    ok = disc >= 0
    sq = torch.sqrt(disc.clamp_min(0))
    q = torch.where(b > 0, -b - sq, -b + sq)
    other = torch.where(q != 0, cc / torch.where(q != 0, q, torch.ones_like(q)), torch.zeros_like(q))
    tin, tout = torch.minimum(q, other), torch.maximum(q, other)
    return ok, tin, tout, _unit(l + tin[:, None] * d), _unit(l + tout[:, None] * d)


def _axes(a):
    return _t([math.cos(a), math.sin(a)]), _t([-math.sin(a), math.cos(a)])


def _halfplanes(o, d, c, edges):
    """Chord of an intersection of half planes (outward normal, a point of the edge), world frame."""
    n = o.shape[0]
    tin, tout = _t([-math.inf]).expand(n).clone(), _t([math.inf]).expand(n).clone()
    nin, nout = torch.zeros_like(o), torch.zeros_like(o)
    ok = torch.ones(n, dtype=torch.bool, device="cuda")
    for nrm, pt in edges:
        num, den = _dot(nrm, (c + pt) - o), _dot(nrm.expand_as(d), d)
        t = num / torch.where(den != 0, den, torch.ones_like(den))
        ok &= (den != 0) | (num >= 0)
        enter, leave = (den < 0) & (t > tin), (den > 0) & (t < tout)
        tin, nin = torch.where(enter, t, tin), torch.where(enter[:, None], nrm, nin)
        tout, nout = torch.where(leave, t, tout), torch.where(leave[:, None], nrm, nout)
    return ok & (tin <= tout), tin, tout, nin, nout


def _edges(obj):
    s, p, _ = obj
    u, v = _axes(p[2])
    if s == "rect":
        hw, hh = 0.5 * p[3], 0.5 * p[4]
        return [(-v, -hh * v), (u, hw * u), (v, hh * v), (-u, -hw * u)]
    pts = [x * u + y * v for x, y in p[3]]
    got = []
    for i, a in enumerate(pts):
        e = pts[(i + 1) % len(pts)] - a
        got.append((_unit(torch.stack([e[1], -e[0]])), a))
    return got


def _lens_centres(p):
    u, _ = _axes(p[2])
    c = _t(p[:2])
    return c + 0.5 * p[4] * u, c - 0.5 * p[4] * u


def _closed_chord(o, d, obj):
    s, p, _ = obj
    if s == "circle":
        return _circle(o, d, _t(p[:2]), p[2])
    if s in ("rect", "poly"):
        return _halfplanes(o, d, _t(p[:2]), _edges(obj))
    if s == "ellipse":
        u, v = _axes(p[2])
        l = o - _t(p[:2])
        os = torch.stack([_dot(l, u.expand_as(l)) / p[3], _dot(l, v.expand_as(l)) / p[4]], 1)
        ds = torch.stack([_dot(d, u.expand_as(d)) / p[3], _dot(d, v.expand_as(d)) / p[4]], 1)
        k = torch.sqrt(_dot(ds, ds))
        ok, tin, tout, _, _ = _circle(os, ds / k[:, None], _t([0.0, 0.0]), 1.0)
        tin, tout = tin / k, tout / k

        def nrm(t):
            x = os + t[:, None] * ds
            return _unit(x[:, :1] / p[3] * u + x[:, 1:] / p[4] * v)

        return ok, tin, tout, nrm(tin), nrm(tout)
    ca, cb = _lens_centres(p)  # a lens: what two circles have in common
    a, b = _circle(o, d, ca, p[3]), _circle(o, d, cb, p[3])
    first, last = a[1] > b[1], a[2] < b[2]
    tin, tout = torch.where(first, a[1], b[1]), torch.where(last, a[2], b[2])
    return (a[0] & b[0] & (tin < tout), tin, tout, torch.where(first[:, None], a[3], b[3]),
            torch.where(last[:, None], a[4], b[4]))


def _curve_hit(o, d, p):
    """Nearest hit of a cubic: f(s) = n . (B(s) - o) has a root in each monotone piece with a change of sign."""
    P = _t(p).reshape(4, 2)
    a3, a2, a1, a0 = -P[0] + 3 * P[1] - 3 * P[2] + P[3], 3 * P[0] - 6 * P[1] + 3 * P[2], 3 * (P[1] - P[0]), P[0]
    n = torch.stack([-d[:, 1], d[:, 0]], 1)
    A, B, C = (_dot(n, x.expand_as(n)) for x in (a3, a2, a1))
    D = _dot(n, a0 - o)
    f = lambda s: ((A * s + B) * s + C) * s + D  # noqa: E731
    disc = (4 * B * B - 12 * A * C).clamp_min(0)
    q = -0.5 * (2 * B + torch.where(B >= 0, 1.0, -1.0) * torch.sqrt(disc))
    r1 = torch.where(A != 0, q / torch.where(A != 0, 3 * A, torch.ones_like(A)), torch.zeros_like(A))
    r2 = torch.where(q != 0, C / torch.where(q != 0, q, torch.ones_like(q)), torch.zeros_like(A))
    k = [torch.zeros_like(A), torch.minimum(r1, r2).clamp(0, 1), torch.maximum(r1, r2).clamp(0, 1), torch.ones_like(A)]
    best, bs = torch.full_like(A, math.inf), torch.zeros_like(A)
    for i in range(3):
        lo, hi = k[i].clone(), k[i + 1].clone()
        sign = f(lo) < 0
        change = (sign != (f(hi) < 0)) & (hi > lo)
        for _ in range(60):
            mid = 0.5 * (lo + hi)
            left = (f(mid) < 0) == sign
            lo, hi = torch.where(left, mid, lo), torch.where(left, hi, mid)
        s = 0.5 * (lo + hi)
        pt = ((a3 * s[:, None] + a2) * s[:, None] + a1) * s[:, None] + a0
        t = _dot(pt - o, d)
        ok = change & (t > T_MIN) & (t < best)
        best, bs = torch.where(ok, t, best), torch.where(ok, s, bs)
    tan = (3 * a3 * bs[:, None] + 2 * a2) * bs[:, None] + a1
    return best, _unit(torch.stack([-tan[:, 1], tan[:, 0]], 1))


def _object_hit(o, d, obj):
    """(t or inf, unit normal)"""
    s, p, _ = obj
    if s == "curve":
        return _curve_hit(o, d, p)
    if s == "mirror":
        a, e = _t(p[:2]), _t(p[2:]) - _t(p[:2])
        den = d[:, 0] * e[1] - d[:, 1] * e[0]
        w = a - o
        inv = 1.0 / torch.where(den != 0, den, torch.ones_like(den))
        t, u = (w[:, 0] * e[1] - w[:, 1] * e[0]) * inv, (w[:, 0] * d[:, 1] - w[:, 1] * d[:, 0]) * inv
        ok = (den != 0) & (t > T_MIN) & (u >= 0) & (u <= 1)
        return torch.where(ok, t, math.inf), _unit(torch.stack([-e[1], e[0]])).expand_as(d)
    ok, tin, tout, nin, nout = _closed_chord(o, d, obj)
    enter = tin > T_MIN
    t = torch.where(enter, tin, tout)
    return torch.where(ok & (t > T_MIN), t, math.inf), torch.where(enter[:, None], nin, nout)


def _contains(pt, obj):
    s, p, _ = obj
    c = _t(p[:2])
    if s == "circle":
        return _dot(pt - c, pt - c) < p[2] * p[2]
    if s == "ellipse":
        u, v = _axes(p[2])
        l = pt - c
        return (_dot(l, u.expand_as(l)) / p[3]) ** 2 + (_dot(l, v.expand_as(l)) / p[4]) ** 2 < 1
    if s == "lens":
        return torch.stack([_dot(pt - x, pt - x) < p[3] * p[3] for x in _lens_centres(p)]).all(0)
    return torch.stack([_dot(pt - (c + e), n.expand_as(pt)) < 0 for n, e in _edges(obj)]).all(0)


def _primary(lights, objs):
    o, d, c, ior = [], [], [], []
    for kind, pos, direction, n, color in lights:
        i = torch.arange(n, dtype=torch.float64, device="cuda")
        x = _t(pos).expand(n, 2)
        if kind == "band":
            e = _t(direction) - _t(pos)
            x = _t(pos) + (i / n)[:, None] * e
            w = _unit(torch.stack([-e[1], e[0]])).expand(n, 2)
        else:
            if kind == "point":
                a, sign = i * 2 * math.pi / n, 1.0
            else:
                spread = _spot_angle(kind)
                mid = math.atan(direction[1] / direction[0])
                a, sign = mid - 0.5 * spread + (i + 1) / n * spread, math.copysign(1.0, direction[0])
            w = sign * torch.stack([torch.cos(a), torch.sin(a)], 1)
        at = 1.0
        for ob in objs:
            if ob[2] is not None and bool(_contains(_t([pos]), ob)[0]):
                at = ob[2]
        o.append(x)
        d.append(w)
        c.append(_t(color).expand(n, 4))
        ior.append(_t([at]).expand(n))
    return [torch.cat(v) for v in (o, d, c, ior)]


def _trace64(scene, bounces, canvas):
    """(positions (S, 4), colours (S, 4)) of every segment in emission order, 64 bits."""
    objs, lights = scene
    o, d, c, ior = _primary(lights, objs)
    key = (torch.arange(o.shape[0], device="cuda") << 24) | 1
    cut = 0.001
    seen = lambda c: ~(((c[:, :3] < cut).all(1)) | (c[:, 3] < cut))  # noqa: E731
    live = seen(c)
    pos, col, keys = [], [], []
    lo, hi = _t([canvas[0], canvas[2]]), _t([canvas[1], canvas[3]])
    for g in range(bounces):
        o, d, c, ior, key = o[live], d[live], c[live], ior[live], key[live]
        if not o.shape[0]:
            break
        best = torch.full_like(ior, math.inf)
        nrm, which = torch.zeros_like(o), torch.full_like(key, -1)
        for k, ob in enumerate(objs):
            t, n = _object_hit(o, d, ob)
            win = t < best
            best, nrm, which = torch.where(win, t, best), torch.where(win[:, None], n, nrm), torch.where(win, k, which)
        hit = which >= 0
        # rays that hit nothing leave through the canvas
        safe = torch.where(d != 0, d, torch.full_like(d, 1e-300))
        ta, tb = (lo - o) / safe, (hi - o) / safe
        t0, t1 = torch.minimum(ta, tb).max(1).values, torch.maximum(ta, tb).min(1).values
        te = torch.where(t0 > T_MIN, t0, t1)
        leaves = (t0 <= t1) & (te > T_MIN)
        t = torch.where(hit, best, te)
        p = o + t[:, None] * d
        emit = hit | leaves
        pos.append(torch.cat([o, p], 1)[emit])
        col.append(c[emit])
        keys.append(key[emit])
        # children
        index = _t([ob[2] if ob[2] is not None else 0.0 for ob in objs] + [0.0])
        closed = torch.tensor([ob[2] is not None for ob in objs] + [False], device="cuda")
        mat = closed[which] & hit
        dn = _dot(d, nrm)
        n2 = index[which]
        out = mat & (dn > 0)
        medium, found = torch.ones_like(n2), torch.zeros_like(out)
        for k, ob in enumerate(objs):
            if ob[2] is not None:
                inside = out & ~found & (which != k) & _contains(p, ob)
                medium, found = torch.where(inside, ob[2], medium), found | inside
        n2 = torch.where(out, medium, n2)
        n2 = torch.where(mat, n2, torch.ones_like(n2))
        nf = torch.where((dn > 0)[:, None], -nrm, nrm)
        ci = dn.abs()
        rd = _unit(d + 2 * ci[:, None] * nf)
        eta = ior / n2
        kk = 1 - eta * eta * (1 - ci * ci)
        through = mat & (kk >= 0)
        ct = torch.sqrt(kk.clamp_min(0))
        td = eta[:, None] * d + (eta * ci - ct)[:, None] * nf
        td = td / torch.sqrt(_dot(td, td)).clamp_min(1e-300)[:, None]
        rs = (ior * ci - n2 * ct) / (ior * ci + n2 * ct)
        rp = (n2 * ci - ior * ct) / (n2 * ci + ior * ct)
        R = torch.where(through, 0.5 * (rs * rs + rp * rp), torch.ones_like(rs))
        one = torch.ones_like(R)
        ca = c * torch.stack([R, R, R, one], 1)
        cb = c * torch.stack([1 - R, 1 - R, 1 - R, one], 1)
        path = (key & 0xFFFFFF) << 1
        ray = key & ~0xFFFFFF
        o = torch.cat([p, p])
        d = torch.cat([rd, td])
        live = torch.cat([hit & seen(ca), through & seen(cb)])
        c = torch.cat([ca, cb])
        ior = torch.cat([ior, n2])
        key = torch.cat([ray | path, ray | path | 1])
    if not pos:
        return torch.zeros((0, 4), dtype=torch.float64, device="cuda"), torch.zeros((0, 4), dtype=torch.float64, device="cuda")
    order = torch.argsort(torch.cat(keys))
    return torch.cat(pos)[order], torch.cat(col)[order]


def _accumulate64(pos, c0, c1, width, height, bounds):
    """The picture of the segments in 64 bits: one sample per major-axis pixel, split between the two
    nearest pixels of the minor axis. None where it would take too long."""
    left, right, bottom, top = bounds
    pos = pos.float().double()  # vertices are 32-bit floats
    sx, sy = width / (right - left), height / (top - bottom)
    X0, Y0, X1, Y1 = (pos[:, 0] - left) * sx, (top - pos[:, 1]) * sy, (pos[:, 2] - left) * sx, (top - pos[:, 3]) * sy
    xm = (X1 - X0).abs() >= (Y1 - Y0).abs()
    M0, M1, m0, m1 = (torch.where(xm, a, b) for a, b in ((X0, Y0), (X1, Y1), (Y0, X0), (Y1, X1)))
    fwd = M1 > M0
    klo = torch.where(fwd, torch.ceil(M0 - 0.5), torch.floor(M1 - 0.5) + 1)
    khi = torch.where(fwd, torch.ceil(M1 - 0.5) - 1, torch.floor(M0 - 0.5))
    limit = torch.where(xm, float(width), float(height))
    klo, khi = klo.clamp_min(0), torch.minimum(khi, limit - 1)
    cnt = torch.where(M1 != M0, (khi - klo + 1).clamp_min(0), torch.zeros_like(klo)).long()
    if int(cnt.sum()) > MOST_SAMPLES:
        return None
    acc = torch.zeros((height * width, 4), dtype=torch.float64, device="cuda")
    ends = torch.cumsum(cnt, 0)
    i = 0
    while i < cnt.numel():
        base = int(ends[i - 1]) if i else 0
        j = max(i + 1, int(torch.searchsorted(ends, torch.tensor(base + 8_000_000, device="cuda"), right=True)))
        n = cnt[i:j]
        who = torch.repeat_interleave(torch.arange(i, min(j, cnt.numel()), device="cuda"), n)
        k = klo[who] + (torch.arange(who.numel(), device="cuda") - (ends[who] - cnt[who] - base)).double()
        s = (k + 0.5 - M0[who]) / (M1[who] - M0[who])
        v = m0[who] + s * (m1[who] - m0[who]) - 0.5
        lo = torch.floor(v)
        f = v - lo
        c = c0[who].double()
        if c1 is not None:
            c = c + s[:, None] * (c1[who].double() - c)
        c = torch.cat([c[:, :3], c[:, 3:] ** 2], 1)
        for m, w in ((lo, 1 - f), (lo + 1, f)):
            x, y = torch.where(xm[who], k, m).long(), torch.where(xm[who], m, k).long()
            ok = (x >= 0) & (x < width) & (y >= 0) & (y < height)
            acc.index_add_(0, (y * width + x)[ok], (c * w[:, None])[ok])
        i = j
    acc = acc.reshape(height, width, 4)
    return {"accum": acc, "image": acc + _t([0.0, 0.0, 0.0, 1.0])}


def _strings64(case, seed):
    pos, c0, c1 = [], [], []
    for m in _strings(case, seed):
        n = m["modulo"]
        i = np.arange(n)
        ix = (i * m["num"]) % n
        ang = i.astype(np.float64) * 2 * math.pi / n
        pt = 0.9 * np.stack([np.cos(ang), np.sin(ang)], 1)

        def color(at):
            s, k = np.zeros((n, 4)), np.zeros(n)
            for mod, rem, col in m["cols"]:
                on = at % mod == rem
                s[on] += np.float32(col)
                k[on] += 1
            return np.where(k[:, None] > 0, s / np.maximum(k, 1)[:, None], np.float32(m["color"]).astype(np.float64))

        pos.append(np.concatenate([pt, pt[ix]], 1))
        c0.append(color(i))
        c1.append(color(ix))
    return _t(np.concatenate(pos)), _t(np.concatenate(c0)), _t(np.concatenate(c1))


def exact(case, seed):
    kind = case["kind"]
    if kind == "frame":
        if case["rays"] > 120000:
            return None
        objs, lights = _scene(case["scene"], case["rays"], case["objects"], random.Random(seed))
        b = _aspect(case["width"], case["height"])
        if case["edit"]:
            objs = [_moved(objs[0])] + objs[1:]
        pos, col = _trace64((objs, lights), case["bounces"], b)
        return _accumulate64(pos, col, None, case["width"], case["height"], b)
    if kind == "trace":
        scene, canvas = _trace_scene(case, seed)
        pos, col = _trace64(scene, case["bounces"], canvas)
        return {"xy": pos.reshape(-1, 2), "rgba": col.repeat_interleave(2, 0)}
    if kind == "strings":
        if case["nested"] or case["points"] * case["mods"] > 500000:
            return None
        pos, c0, c1 = _strings64(case, seed)
        return _accumulate64(pos, c0, c1 if case["colors"] else None, case["width"], case["height"],
                             _aspect(case["width"], case["height"]))
    if kind == "lines":
        pos, c0, c1, b = _lines(case, seed)
        return _accumulate64(torch.from_numpy(pos).cuda(), torch.from_numpy(c0).cuda(),
                             None if c1 is None else torch.from_numpy(c1).cuda(), case["width"], case["height"], b)
    got = []  # the smaller scenes of a batch or burst
    for i, ((objs, lights), bounces, side) in enumerate((_batch_scenes if kind == "batch" else _serve_scenes)(case, seed)):
        r = None
        if sum(l[3] for l in lights) <= 20000 and len(got) < 12:
            if kind == "serve" and i % 3 == 0:
                objs = [_moved(objs[0])] + objs[1:]
            pos, col = _trace64((objs, lights), bounces, BOUNDS)
            r = _accumulate64(pos, col, None, side, side, BOUNDS)
        got.append(r if r is not None else {"accum": None, "image": None})
    return got
