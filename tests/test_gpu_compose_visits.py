"""How a recorded call is applied to a window of a canvas row (one record or
several, up to 64 runs or more, narrower than 64 pixels or not, cut by window
borders, every blend mode), against the oracle and the per-call form: equal byte
for byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import pixie_amd as px
    px.init()
    return px


def comb(x0, x1, y0, y1, n):
    """A closed zigzag of n teeth from x0 to x1."""
    x = np.linspace(x0, x1, 2 * n + 1)
    y = np.where(np.arange(2 * n + 1) % 2 == 0, y1, y0)
    return "M " + " L ".join("%.3f %.3f" % p for p in zip(x, y)) + " Z"


def rect(x, y, w, h):
    return "M %s %s h %s v %s h %s Z" % (x, y, w, h, -w)


# from below, at and above 64 pixels; at and across the 512-pixel windows
SPANS = [(3.5, 20), (0, 64), (1, 63), (2.25, 61), (5, 60), (6, 64.5), (447.5, 64), (448, 63.5), (500, 30.25),
         (511.5, 1), (512, 60), (509, 66), (900, 600), (1000, 24), (1020, 20), (-5.5, 40), (-600, 2000)]


def both(px, orc, w, h, calls, a8=False):
    rng = np.random.default_rng(w)
    back = rng.integers(0, 256, (h, w) if a8 else (h, w, 4), dtype=np.uint8)
    if not a8:  # premultiplied, with clear and opaque parts
        back[:, : w // 4, 3] = 255
        back[:, w // 4: w // 2, 3] = 0
        back[..., :3] = np.minimum(back[..., :3], back[..., 3:])
    one, two = px.Image.from_array(back), px.Image.from_array(back)
    want = np.repeat(back[..., None], 4, 2) if a8 else back.copy()
    sc = px.Scene()
    for path, kw in calls:
        orc.fill_path(want, path, kw["color"], winding=kw.get("windingRule", 0), mode=kw.get("blendMode", 0))
        one.fillPath(path, **kw)
        sc.fillPath(path, **kw)
    sc.render(two)
    a, b = one.download(), two.download()
    assert np.array_equal(a, b), "%d of %d bytes differ" % ((a != b).sum(), a.size)
    want = want[..., 3] if a8 else want
    assert np.array_equal(a, want), "%d of %d bytes differ from the oracle" % ((a != want).sum(), a.size)


@pytest.mark.parametrize("w", [1023, 1024, 61])
@pytest.mark.parametrize("mode", range(20))
def test_spans(gpu, orc, mode, w):
    rng = np.random.default_rng(mode)
    calls = []
    for i, (x, n) in enumerate(SPANS):
        color = tuple(int(v) for v in rng.choice([0, 1, 77, 128, 200, 254, 255], 4))
        for path in (rect(x, 2 + i % 3, n, 9), comb(x, x + n, 3.3, 12.6, 1 + int(abs(n)) // 9)):
            calls.append((path, dict(color=color, blendMode=mode, windingRule=i & 1)))
    both(gpu, orc, w, 17, calls)


@pytest.mark.parametrize("n", [10, 31, 32, 33, 70, 200])
def test_many_runs(gpu, orc, n):
    both(gpu, orc, 1300, 24, [(comb(x, x + 300, 2.2, 20.7, n), dict(color=(80, 20, 200, 190))) for x in (4, 350.5, 900)])


def test_a8(gpu, orc):
    both(gpu, orc, 1023, 17, [(rect(x, 2, n, 9), dict(color=(9, 9, 9, 150))) for x, n in SPANS], a8=True)
