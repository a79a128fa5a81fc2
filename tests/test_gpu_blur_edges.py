"""Blur, spread and shadow at the edges of their kernels' tiles and radius
classes, against the oracle: equal byte for byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import pixie_amd as px
    px.init()
    return px


@pytest.fixture(scope="module")
def orc():
    import oracle
    return oracle


def picture(w, h, seed):
    """Straight noise, then flat bright and transparent blocks (the largest and
    smallest sums)."""
    rng = np.random.default_rng(seed)
    a = rng.integers(0, 256, (h, w, 4), dtype=np.uint8)
    a[: h // 2, : w // 3] = 255
    a[h // 3:, w // 2:] = np.where(rng.random((h - h // 3, w - w // 2, 1)) < 0.5, 0, a[h // 3:, w // 2:])
    a[..., :3] = np.minimum(a[..., :3], a[..., 3:])
    return a


SIZES = [(1, 1), (2, 63), (3, 5), (47, 49), (48, 48), (64, 64), (65, 33), (97, 193), (195, 130), (256, 70)]
PLANES = SIZES + [(1040, 520), (1041, 517)]  # and beyond the small alpha planes


@pytest.mark.parametrize("w,h", SIZES)
@pytest.mark.parametrize("r", [1, 2, 7, 8, 9, 15, 16, 17, 24, 25, 32, 33, 40, 70])
def test_blur(gpu, orc, r, w, h):
    a = picture(w, h, r)
    want = a.copy()
    orc.blur(want, r, (40, 0, 9, 77))
    img = gpu.Image.from_array(a)
    img.blur(r, (40, 0, 9, 77))
    assert np.array_equal(img.download(), want)


@pytest.mark.parametrize("w,h", PLANES)
@pytest.mark.parametrize("s", [1, 2, 3, 4, 5, 8, 31, 300, -1, -2, -7, -300])
def test_spread(gpu, orc, s, w, h):
    a = picture(w, h, abs(s))
    want = a.copy()
    orc.spread(want, s)
    img = gpu.Image.from_array(a)
    img.spread(s)
    assert np.array_equal(img.download(), want)


@pytest.mark.parametrize("w,h", PLANES)
@pytest.mark.parametrize("offset,spread,blur", [((0, 0), 0, 0), ((1, -2), 0, 1), ((7, 3), 3, 0), ((-5, 2), 2, 8),
                                                ((2.5, -5.25), 0, 16), ((64, 1), -2, 17), ((0, 3), 1, 24),
                                                ((2, 2), 5, 40), ((3, 900), 1, 2)])
def test_shadow(gpu, orc, offset, spread, blur, w, h):
    a = picture(w, h, blur)
    color = (9, 120, 30, 200)
    got = gpu.Image.from_array(a).shadow(offset, spread, blur, color).download()
    assert np.array_equal(got, orc.shadow(a, offset, spread, blur, color))


def test_largest_radius(gpu, orc):
    a = picture(65, 133, 5)
    want = a.copy()
    orc.blur(want, 276, (1, 2, 3, 4))
    img = gpu.Image.from_array(a)
    img.blur(276, (1, 2, 3, 4))
    assert np.array_equal(img.download(), want)
    assert np.array_equal(img.shadow((1, 1), 0, 276, (9, 9, 9, 99)).download(),
                          orc.shadow(want, (1, 1), 0, 276, (9, 9, 9, 99)))
    for call in (lambda: img.blur(277), lambda: img.shadow((1, 1), 0, 277, (9, 9, 9, 99))):
        with pytest.raises(gpu.PixieError) as e:
            call()
        assert e.value.code == 9
    assert np.array_equal(img.download(), want)
