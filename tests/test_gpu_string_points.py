"""StringMods that take their curve's points from a table (draws of 4096 segments and more) give the
segments of those that compute them, bit for bit: every curve, shared and different curves, a
modulo colour, a nested StringMod beside them, and a draw just below and at the border."""
import numpy as np
import pytest

import light_garden_amd as lg
from light_garden_amd import string_mod
from light_garden_amd.string_mod import ModRemColor, StringMod

pytestmark = pytest.mark.gpu


def mods():
    kw = dict(modulo=487, scale=0.9, color=(0.01, 0.02, 0.03, 0.5))
    return [StringMod(num=2, **kw), StringMod(num=77, **kw),
            StringMod(num=3, turns=2, modulo_colors=[ModRemColor(3, 1, (0.5, 0.1, 0.2, 0.9))], **kw),
            StringMod.complex_exp(complex(0.99, 0.02), num=5, **kw),
            StringMod.hypotrochoid(3, 7, 2, num=4, **kw), StringMod.lissajous(3, 4, 0.3, num=9, **kw),
            StringMod(modulo=29, num=3, scale=0.9, nested=StringMod(modulo=400, num=7))]


def drawn(ctx, ms):
    segs = lg.Segments(ctx, vertex_colors=True)
    n = string_mod.draw(ctx, ms, segs)
    return n, segs.download()


@pytest.mark.parametrize("filler", [4096 - 3322 - 1, 4096 - 3322, 60000])
def test_table_equals_own_points(ctx, filler):
    n, alone = drawn(ctx, mods())
    assert n == 6 * 487 + 400 < 4096
    m, more = drawn(ctx, mods() + [StringMod(modulo=filler, num=2)])
    assert m == n + filler
    for a, b in zip(alone, more):
        np.testing.assert_array_equal(a, b[:n])
