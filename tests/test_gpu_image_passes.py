"""Image passes at the edges of their tiles and vectors, against the oracle:
transformed draws over long rows (the running sums of positions from run to run,
tiles cut by spans and borders), integer draws at every offset within a vector,
opacities, and per-call fills by the width of their windows.  All equal byte for
byte."""
import math

import numpy as np
import pytest

import pixie_amd as px
from test_oracle_draw import T, S, R, mul

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    px.init()
    return px


def picture(seed, w, h):
    rng = np.random.default_rng(seed)
    a = rng.integers(0, 256, (h, w, 4), dtype=np.uint8)
    a[..., :3] = np.minimum(a[..., :3], a[..., 3:4])
    a[rng.random((h, w)) < 0.2] = 0
    return a


MATS = [mul(T(60, -300), R(math.radians(30))), mul(T(2600, 5), R(math.radians(171))), mul(T(3, 2.5), S(3.7, 1.01)),
        mul(T(-1000.3, 0.25), S(0.9999, 0.37)), mul(T(100, 1), S(60.0, 0.5)), mul(T(2500, 20), S(-3.3, -0.7)),
        mul(T(1300, -40), mul(R(math.radians(89.9)), S(2.2, 1.1))), mul(T(15.5, 0.5), S(1.0, 1.0)),
        mul(T(511.7, 3), S(0.25, 0.25))]


@pytest.mark.parametrize("mode", [0, 1, 16, 17])
@pytest.mark.parametrize("k", range(len(MATS)))
def test_long_rows(gpu, orc, k, mode):
    base, b = picture(k, 2611, 39), picture(k + 50, 700, 450)
    img = px.Image.from_array(base)
    img.draw(px.Image.from_array(b), transform=MATS[k], blendMode=mode)
    want = base.copy()
    orc.draw_transform(want, b, MATS[k], mode)
    assert np.array_equal(img.download(), want)


@pytest.mark.parametrize("a8", [False, True])
@pytest.mark.parametrize("mode", [0, 1, 4, 16, 17, 18])
def test_offsets(gpu, orc, mode, a8):
    for w, h, bw, bh in ((9, 3, 6, 2), (16, 3, 16, 3), (5, 5, 11, 9), (1, 1, 2, 2), (1030, 2, 1027, 2)):
        base, b = picture(w, w, h), picture(bw + 9, bw, bh)
        if a8:
            b = np.repeat(b[..., 3:], 4, axis=2)
        for dx in (-7, -4, -3, -1, 0, 1, 2, 3, 4, 6):
            for dy in (-1, 0, 2):
                img = px.Image.from_array(base)
                img.draw(px.Image.from_array(b[..., 0].copy() if a8 else b), dx, dy, mode)
                want = base.copy()
                orc.draw(want, b, dx, dy, mode)
                assert np.array_equal(img.download(), want), (w, h, bw, bh, dx, dy)


@pytest.mark.parametrize("o", [0.002, 0.3, 0.5, 0.998, 1.7])
def test_opacity(gpu, orc, o):
    for w, h in ((1, 1), (3, 1), (1025, 3)):
        a = picture(w, w, h)
        want = a.copy()
        orc.apply_opacity(want, o)
        img = px.Image.from_array(a)
        img.applyOpacity(o)
        assert np.array_equal(img.download(), want)


@pytest.mark.parametrize("teeth", [0, 1, 12, 31, 32, 33, 60])
@pytest.mark.parametrize("w,h", [(500, 3300), (1537, 3100), (2049, 3100), (3300, 1600)])
def test_window_widths(gpu, orc, w, h, teeth):
    """Per-call fills in windows of 512 to 1,536 px, of few and many entries a
    row, against the oracle and the recorded form (windows of 512 px)."""
    d = "M 5.5 3 L %s 2.25 Q %s %s %s %s L 2 %s Z" % (w - 4, w - 1, h / 2, w - 9.5, h - 3, h - 1.5)
    for k in range(teeth):
        x = 20 + k * (w - 60) / teeth
        d += " M %.2f %.2f L %.2f %.2f L %.2f %.2f Z" % (x, h - 9.3, x + 3.3, 11.1 + k, x + 9.7, h - 20.2)
    for mode, color in ((0, (30, 200, 90, 180)), (16, (255, 255, 255, 255))):
        base = picture(7, w, h)
        img = px.Image.from_array(base)
        img.fillPath(d, color, blendMode=mode, windingRule=1)
        sc = px.Scene()
        sc.fillPath(d, color, blendMode=mode, windingRule=1)
        two = px.Image.from_array(base)
        sc.render(two)
        got, want = img.download(), base.copy()
        assert np.array_equal(got, two.download())
        orc.fill_path(want, d, color, winding=1, mode=mode)
        assert np.array_equal(got, want)
