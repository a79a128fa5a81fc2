"""Rows by the number of entries that they select, at the edges of the forms that
walk them (8, 16, 32 and 64 lanes a sample line, register slots, the LDS stage,
presorted rows, a workgroup per row): the per-call and the recorded form against
the oracle, byte for byte.  The shapes have what the walks tell apart: slivers
within a pixel, hits at one x whose windings cancel or add up, hits on pixel and
window borders, and hits left and right of the canvas."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W, H = 1150, 21


@pytest.fixture(scope="module")
def gpu():
    import pixie_amd as px
    px.init()
    return px


def quad(x, y0, y1, width, slope):
    """A thin parallelogram: two edges on each of its rows."""
    d = slope * (y1 - y0)
    return [(x, y0), (x + width, y0), (x + width + d, y1), (x + d, y1)]


def slivers(rng, n):
    out = []
    for _ in range(n // 2):
        y0 = rng.uniform(0.2, 4.8)
        out.append(quad(rng.uniform(-6, W + 4), y0, y0 + rng.uniform(9, 15), rng.choice([0.02, 0.1, 0.4, 0.9, 1.7]),
                        rng.uniform(-0.6, 0.6)))
    return out


def stacks(rng, n):
    """Boxes that share their edges' x, drawn both ways round."""
    out = []
    xs = np.concatenate([[0.0, 0.5, 64.0, 255.75, 511.5, 512.0, 512.25, 1023.5, 1024.0, W - 1.0, W], rng.uniform(0, W, 6)])
    for k in range(n // 2):
        a, b = np.sort(rng.choice(xs, 2, replace=False))
        y0 = rng.uniform(0.2, 4.8)
        q = quad(a, y0, y0 + rng.uniform(9, 15), b - a, 0.0)
        out.append(q if k % 3 else q[::-1])
    return out


def zigzag(rng, n):
    """One contour whose edges cross each other inside rows."""
    y = np.where(np.arange(n) % 2 == 0, rng.uniform(0.3, 4, n), rng.uniform(14, 20, n))
    return [list(zip(rng.uniform(-20, W + 20, n), y))]


SIZES = [2, 4, 6, 8, 10, 16, 18, 32, 34, 62, 64, 66, 128, 130, 254, 256, 258, 510, 512, 514, 700, 1024, 1026, 1300, 2600]


@pytest.mark.parametrize("rule", [0, 1])
@pytest.mark.parametrize("kind", [slivers, stacks, zigzag])
@pytest.mark.parametrize("n", SIZES)
def test_row_walks(gpu, orc, n, kind, rule):
    rng = np.random.default_rng(n)
    cmds = []
    for shape in kind(rng, n):
        for i, (x, y) in enumerate(shape):
            cmds += [1.0 if i == 0 else 2.0, x, y]
        cmds.append(0.0)
    cmds = np.array(cmds, np.float32)
    color = (180, 90, 30, 210)
    back = rng.integers(0, 256, (H, W, 4), dtype=np.uint8)
    back[..., :3] = np.minimum(back[..., :3], back[..., 3:])
    want = back.copy()
    orc.fill_path(want, cmds, color, winding=rule)
    one, two = gpu.Image.from_array(back), gpu.Image.from_array(back)
    one.fillPath(cmds, color, windingRule=rule)
    sc = gpu.Scene()
    sc.fillPath(cmds, color, windingRule=rule)
    sc.render(two)
    for what, img in (("per call", one), ("recorded", two)):
        got = img.download()
        bad = np.argwhere((got != want).any(2))
        assert len(bad) == 0, "%s: %d pixels, first %s got %s want %s" % (
            what, len(bad), bad[0], got[tuple(bad[0])], want[tuple(bad[0])])
