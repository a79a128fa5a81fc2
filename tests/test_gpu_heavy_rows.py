"""Rows of bands with hundreds of entries in the batched form (the workgroup
row kernel) against the oracle and against the per-call form, which runs the
one-wave row program on the same shapes: the images must be equal byte for byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import pixie_amd as px
    px.init()
    return px


def teeth(n, x0, x1, y0, y1, jitter=0.0, seed=0):
    """A closed zigzag of n teeth between y0 and y1: 2n steep edges per row."""
    rng = np.random.default_rng(seed)
    x = np.linspace(x0, x1, 2 * n + 1) + (rng.uniform(-jitter, jitter, 2 * n + 1) if jitter else 0)
    y = np.where(np.arange(2 * n + 1) % 2 == 0, y1, y0) + rng.uniform(-0.3, 0.3, 2 * n + 1)
    return np.stack([x, y], 1).astype(np.float32)


def shape_cmds(shapes):
    out = []
    for s in shapes:
        for i, (x, y) in enumerate(s):
            out += [1.0 if i == 0 else 2.0, x, y]
        out.append(0.0)
    return np.array(out, np.float32)


def closed(shapes):
    return [np.concatenate([s, s[:1]]) for s in shapes]


def both(px, orc, shapes, w, h, rule, mode, a8=False):
    color = (200, 90, 30, 220)
    back = np.random.default_rng(1).integers(0, 256, (h, w) if a8 else (h, w, 4), dtype=np.uint8)
    if not a8:
        back[..., :3] = np.minimum(back[..., :3], back[..., 3:])
    want = np.repeat(back[..., None], 4, 2) if a8 else back.copy()
    orc.fill_path(want, shape_cmds(shapes), color, winding=rule, mode=mode)
    want = want[..., 3] if a8 else want
    one, two = px.Image.from_array(back), px.Image.from_array(back)
    one.fillShapes(closed(shapes), color, windingRule=rule, blendMode=mode)
    sc = px.Scene()
    sc.fillPath(shape_cmds(shapes), color, windingRule=rule, blendMode=mode)
    sc.render(two)
    a, b = one.download(), two.download()
    assert np.array_equal(a, b), "%d of %d bytes differ" % ((a != b).sum(), a.size)
    assert np.array_equal(a, want), "%d of %d bytes differ from the oracle" % ((a != want).sum(), a.size)
    two.upload(back)
    sc.render(two)  # a replay
    assert np.array_equal(a, two.download())


def cases():
    rng = np.random.default_rng(3)
    # hits per 64-px bucket of one register slot, of four, beyond four, and
    # more hits in a line than the key space (left to the rows kernel)
    for n, width in ((520, 3000), (600, 640), (700, 300), (900, 100), (4000, 2000)):
        yield "teeth%d_w%d" % (n, width), [teeth(n, 7.3, 7.3 + width, 3, 40, 0.4, n)], 3100, 48
    # bucket and window borders: edges at whole multiples of 64 px
    comb = [np.array([[64 * k, 2], [64 * k, 30.5], [64 * k + 32, 29.7], [64 * k + 32.5, 2.2]], np.float32)
            for k in range(48)] * 6
    yield "borders", comb, 3072, 36
    # one contour many times over, both ways round: equal x, cancelling pairs
    ring = teeth(60, 20, 600, 4, 28, 0.2, 9)
    yield "cancel", [ring, ring[::-1]] * 6 + [ring], 640, 32
    # teeth left of the canvas, right of it, and across both borders
    yield "clipped", [teeth(700, -900, 2100, 2, 30, 1.0, 4)], 1023, 33
    # several window groups, and a ragged last window
    yield "wide", [teeth(2500, 10, 5003, 2, 20, 0.5, 5)], 5007, 23
    # random stars
    yield "stars", [rng.uniform(0, 500, (40, 2)).astype(np.float32) for _ in range(40)], 517, 509


@pytest.mark.parametrize("rule", [0, 1])
@pytest.mark.parametrize("name,shapes,w,h", list(cases()), ids=[c[0] for c in cases()])
def test_heavy_rows(gpu, orc, name, shapes, w, h, rule):
    both(gpu, orc, shapes, w, h, rule, 0)


@pytest.mark.parametrize("mode", [16, 17])
def test_heavy_rows_mask_and_overwrite(gpu, orc, mode):
    both(gpu, orc, [teeth(600, 30, 2500, 3, 40, 0.4, 1)], 2600, 48, 0, mode)


def test_heavy_rows_a8(gpu, orc):
    both(gpu, orc, [teeth(600, 30, 2500, 3, 40, 0.4, 1)], 2600, 48, 0, 0, a8=True)


def test_heavy_rows_sample_lines_through_vertices(gpu, orc):
    # beyond y = 4096 float32 rounds the middle sample line onto y + 0.5, so
    # vertices there count twice and a line's windings do not sum to 0
    z = teeth(600, 10, 900, 4100, 4140, 0.0, 2)
    z[:, 1] = np.floor(z[:, 1]) + 0.5
    mid = z.copy()
    mid[::2, 1] -= 20.0
    both(gpu, orc, [z, mid], 950, 4160, 0, 0)


def test_profile_names_each_row_kernel(gpu):
    sc, img = gpu.Scene(), gpu.Image(2600, 48)
    sc.fillPath(shape_cmds([teeth(600, 30, 2500, 3, 40, 0.4, 1)]), (200, 90, 30, 220))
    sc.render(img)
    gpu.profile_begin()
    sc.render(img)
    gpu.profile_end()
    for name in ("scene_heavy_kernel", "scene_rows_kernel"):
        ms, launches = gpu.profile_kernel(name)
        assert launches == 1 and ms > 0, (name, ms, launches)
