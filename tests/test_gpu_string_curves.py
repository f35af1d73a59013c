"""One call over many StringMods: the segments of each equal the StringMod drawn alone, bit for bit,
with curves that differ in one parameter each and come back later in the call; the call's time grows
with the number of StringMods, not with its square, and is the same whether they share a curve."""
import ctypes as C
import time

import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import abi, string_mod

pytestmark = pytest.mark.gpu


def curves():
    base = dict(modulo=331, num=3, turns=1, scale=0.9)
    other = [dict(modulo=332), dict(turns=2), dict(scale=0.8), dict(num=5),
             dict(curve=string_mod.CURVE_COMPLEX_EXP, curve_f=(0.5, 0.5)), dict(curve=string_mod.CURVE_COMPLEX_EXP, curve_f=(0.5, 0.6)),
             dict(curve=string_mod.CURVE_HYPOTROCHOID, curve_u=(5, 3, 2)), dict(curve=string_mod.CURVE_HYPOTROCHOID, curve_u=(5, 3, 1)),
             dict(curve=string_mod.CURVE_LISSAJOUS, curve_u=(3, 2, 0), curve_f=(0.25, 0.0))]
    return [base] + [dict(base, **o) for o in other]


def test_shared_curves_equal_single_draws(ctx):
    params = curves()
    order = list(range(len(params))) + list(range(len(params)))[::-1] + [0, 0, 3]
    mods = [lg.StringMod(color=[0.001 * (i + 1)] * 4, **params[k]) for i, k in enumerate(order)]
    segs, one = lg.Segments(ctx, vertex_colors=True), lg.Segments(ctx, vertex_colors=True)
    string_mod.draw(ctx, mods, segs)
    pos, c0, c1, _ = segs.download()
    assert len(pos) >= 4096
    at = 0
    for m in mods:
        n = string_mod.draw(ctx, [m], one)
        p, a, b, _ = one.download()
        np.testing.assert_array_equal(pos[at:at + n], p)
        np.testing.assert_array_equal(c0[at:at + n], a)
        np.testing.assert_array_equal(c1[at:at + n], b)
        at += n
    assert at == len(pos)


def test_time_grows_with_the_curves(ctx):
    segs = lg.Segments(ctx, vertex_colors=True)

    def call(n):
        mods = [lg.StringMod(modulo=20 + i % 7, num=2, scale=0.9 - 1e-6 * i, color=[0.001] * 4) for i in range(n)]
        arr, keep = (abi.LgStringMod * n)(), []
        for i, m in enumerate(mods):
            arr[i], k = m.to_abi()
            keep.append(k)
        best = 1e9
        for _ in range(6):
            t = time.perf_counter()
            abi.call("lg_string_mod_draw", ctx.handle, n, arr, segs.handle)
            best = min(best, time.perf_counter() - t)
        return best

    few, many = call(3000), call(24000)
    print("3000 curves %.2f ms, 24000 curves %.2f ms" % (1e3 * few, 1e3 * many))
    assert many < 16 * few + 2e-3  # eight times the work


def test_curves_need_not_be_shared(ctx):
    segs = lg.Segments(ctx, capacity=1_700_000, vertex_colors=True)
    best = {}
    calls = {}
    for name, step in (("shared", 0), ("own", 1)):
        arr, keep = (abi.LgStringMod * 16)(), []
        for i in range(16):
            arr[i], k = lg.StringMod(modulo=100000 + step * i, num=2 + i, scale=0.9, color=[0.001] * 4).to_abi()
            keep.append(k)
        calls[name] = (arr, keep)
    for _ in range(60):
        for name, (arr, _) in calls.items():
            t = time.perf_counter()
            abi.call("lg_string_mod_draw", ctx.handle, 16, arr, segs.handle)
            best[name] = min(best.get(name, 1.0), time.perf_counter() - t)
    print("16 x 100000 points: one curve %.1f us, 16 curves %.1f us" % (1e6 * best["shared"], 1e6 * best["own"]))
    assert best["own"] < 1.25 * best["shared"]
