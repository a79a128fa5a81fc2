"""The batched form's splits of its work (lanes per command, lanes per stroke
point and chunks of points, calls per planning workgroup, bands per tile)
at their edges, against the oracle and the per-call form: equal byte for byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import pixie_amd as px
    px.init()
    return px


def curves(n, w, h, seed):
    """A contour of n commands after its move: lines, cubics, quads, arcs."""
    rng = np.random.default_rng(seed)
    p = lambda: "%.2f %.2f" % (rng.uniform(2, w - 2), rng.uniform(2, h - 2))
    d = ["M " + p()]
    for i in range(n):
        k = int(rng.integers(0, 5))
        d.append({0: "L " + p(), 1: "C %s %s %s" % (p(), p(), p()), 2: "Q %s %s" % (p(), p()), 3: "S %s %s" % (p(), p()),
                  4: "A %.1f %.1f 20 %d %d %s" % (rng.uniform(5, 60), rng.uniform(5, 60), i & 1, (i >> 1) & 1, p())}[k])
    return " ".join(d)


def both(px, orc, w, h, calls, exact=True):
    one, two = px.Image(w, h), px.Image(w, h)
    want = orc.new_image(w, h)
    sc = px.Scene()
    for kind, path, kw in calls:
        getattr(one, kind)(path, **kw)
        getattr(sc, kind)(path, **kw)
        if kind == "fillPath":
            orc.fill_path(want, path, kw["color"], winding=kw.get("windingRule", 0))
        else:
            orc.stroke_path(want, px.parse_path(path), kw["color"], width=kw["strokeWidth"], cap=kw.get("lineCap", 0),
                            join=kw.get("lineJoin", 0), dashes=kw.get("dashes", ()))
    sc.render(two)
    a, b = one.download(), two.download()
    assert np.array_equal(a, b), "%d of %d bytes differ" % ((a != b).sum(), a.size)
    d = np.abs(a.astype(int) - want).max(2)
    # Hits at one x on a row whose edges all span it, but not as trapezoids: pixie
    # takes them in the order of the edges' middles, a row of at most 64 entries
    # here in the order of the band.  A span may then be cut in two, each part
    # rounded down: the bar of the path tests.
    assert d.max() <= (0 if exact else 1) and (d > 0).mean() <= 1e-4, "%d pixels differ from the oracle" % (d > 0).sum()
    two.upload(np.zeros((h, w, 4), np.uint8))
    sc.render(two)  # a replay
    assert np.array_equal(a, two.download())


@pytest.mark.parametrize("n", [1, 30, 31, 32, 33, 62, 63, 64, 65, 126, 127, 128, 129, 255, 256, 257])
def test_lanes_per_command(gpu, orc, n):
    d = curves(n, 300, 200, n)
    calls = [("fillPath", d, dict(color=(200, 40, 90, 200), windingRule=n & 1)),
             ("strokePath", d, dict(color=(20, 140, 90, 150), strokeWidth=2.5, lineJoin=n % 3))]
    both(gpu, orc, 300, 200, calls[:1])
    both(gpu, orc, 300, 200, calls, exact=False)


@pytest.mark.parametrize("style", [dict(), dict(lineJoin=1), dict(lineCap=1), dict(lineCap=2, lineJoin=2),
                                   dict(lineJoin=1, lineCap=1, dashes=[9.0, 3.5])],
                         ids=["miter", "round", "caps", "bevel", "dashed"])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 255, 256, 257, 513])
def test_stroke_chunks(gpu, orc, n, style):
    rng = np.random.default_rng(n)
    x = np.linspace(5, 395, n)
    y = 60 + 40 * np.sin(x / 23) + rng.uniform(-4, 4, n)
    d = "M " + " L ".join("%.2f %.2f" % q for q in zip(x, y))
    both(gpu, orc, 400, 120, [("strokePath", d + z, dict(color=(90, 40, 190, 180), strokeWidth=3.0, **style))
                         for z in ("", " Z")])


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1025, 4095, 4096, 4097, 9001])
def test_calls_and_bands(gpu, orc, n):
    rng = np.random.default_rng(n)
    calls = []
    for i in range(n):
        x, y = rng.uniform(-4, 250), rng.uniform(-4, 120)
        w, h = rng.uniform(2, 12, 2)
        d = "M %.2f %.2f l %.2f %.2f l %.2f %.2f z" % (x, y, w, h, -w, h * 0.3)
        calls.append(("fillPath", d, dict(color=tuple(int(v) for v in rng.integers(0, 256, 4)))))
    both(gpu, orc, 256, 128, calls)
