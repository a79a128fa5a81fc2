"""Fills on a canvas wider than 2^23 pixels, where a 24.8 position leaves 32
bits: pixie keeps such a hit as the lowest 32-bit number, so it counts as lying
left of every pixel.  Both forms against the oracle, byte for byte (the oracle
leaves out what pixie then writes beyond the path's columns)."""
import numpy as np
import pytest

import pixie_amd as px

pytestmark = pytest.mark.gpu

W, H, LIMIT = 8_390_000, 2, 1 << 23


def polygon(points):
    out = []
    for i, (x, y) in enumerate(points):
        out += [1.0 if i == 0 else 2.0, x, y]
    return np.array(out + [0.0], np.float32)


def bar(x0, x1):
    """Edges that end inside their row, as all here: no row is a trapezoid."""
    return polygon([(x0, 0.25), (x1, 0.3), (x1 - 40, 0.9), (x0 + 40, 0.85)])


def comb(x0, x1, n):
    """2n edges of slopes either way."""
    x = np.linspace(x0, x1, 2 * n + 1)
    return polygon([(a, 1.15 if i % 2 else 1.8) for i, a in enumerate(x)])


# the selection of a row: at most 8 entries, one register slot, several slots,
# more than the register slots hold
SHAPES = {
    "across": bar(100, LIMIT + 842),
    "beyond": bar(LIMIT + 200, LIMIT + 900),
    "at": bar(LIMIT - 400, LIMIT + 300),
    "below": bar(LIMIT - 900, LIMIT - 100),
    "comb20": comb(LIMIT - 1500, LIMIT + 1300, 20),
    "comb100": comb(LIMIT - 1500, LIMIT + 1300, 100),
    "comb180": comb(LIMIT - 1500, LIMIT - 60, 180),
    "comb300": comb(LIMIT - 1500, LIMIT + 1300, 300),
}


@pytest.mark.parametrize("rule", [0, 1])
@pytest.mark.parametrize("name", list(SHAPES))
def test_wide_canvas(orc, name, rule):
    px.init()
    path, color = SHAPES[name], (200, 90, 30, 220)
    want = orc.new_image(W, H)
    orc.fill_path(want, path, color, winding=rule)
    img = px.Image(W, H)
    img.fillPath(path, color, windingRule=rule)
    assert np.array_equal(img.download(), want), "per call"
    sc = px.Scene()
    sc.fillPath(path, color, windingRule=rule)
    two = px.Image(W, H)
    sc.render(two)
    assert np.array_equal(two.download(), want), "recorded"
