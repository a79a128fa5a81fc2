"""The drawing work that programs have pixie_amd do, as timed cases.

A case is a plain dict; `prepare` makes what a program holds before the call
(canvases, images, recorded scenes, loaded fonts, parsed documents), `run` is
one pass through the public entry points and `work` says what the pass cannot
do without.  Sizes are those of the repository's workloads and tests (the
512-px star, the mixed scene and the glyph atlas of workloads.py, the text
page and paragraph, the 900-px document, the 4096-px image operations) and odd
ones between them.

Every output is the image itself, in bytes.  Coverage, blends and blurs are
integer arithmetic on float32 geometry whose operation order pixie fixes, so
another correct implementation gives the same bytes: all tolerances are
"exact", and no output is a float that 64 bits would refine.
"""
import math
import os

import numpy as np
import torch

import pixie_amd as px

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FONTS = {"noto": "NotoSans-Regular_4.ttf", "roboto": "Roboto-Regular_1.ttf",
         "ubuntu": "Ubuntu-Regular_1.ttf", "inter": "Inter-Regular.ttf"}
CLOSE, MOVE, LINE, CUBIC, QUAD = 0.0, 1.0, 2.0, 5.0, 7.0


def listed():
    return [
        # The smallest call: one opaque fill of a 64-point star.
        {"name": "star_512", "kind": "fill", "w": 512, "h": 512, "points": 64, "mode": 0},
        # A user-interface frame drawn call by call, as code written against
        # pixie draws it: panels, blobs, dashed outlines, gradient buttons.
        {"name": "frame_1280x720", "kind": "frame", "w": 1280, "h": 720, "ops": 24},
        # Four requests of a serving loop: each records its scene, renders it
        # on its own execution lane and blurs it if asked.
        {"name": "serve_4_lanes", "kind": "serve", "side": 701, "paths": 24, "blur": 8},
        # A small recorded scene drawn again each frame.
        {"name": "scene_1023x767", "kind": "scene", "w": 1023, "h": 767, "paths": 100},
        # The mixed fill + stroke scene: 2,000 paths on 4096 x 4096.
        {"name": "scene_4096", "kind": "scene", "w": 4096, "h": 4096, "paths": 2000},
        # A glyph atlas: 10,000 outlines into one 8-bit image.
        {"name": "atlas_8192", "kind": "atlas", "w": 8192, "glyphs": 10000},
        # A paragraph laid out and drawn in one call.
        {"name": "paragraph_1000x150", "kind": "text", "w": 1000, "h": 150, "font": "roboto",
         "size": 16, "words": 150, "typeset": True},
        # A page of 33,000 glyphs whose layout the program keeps.
        {"name": "page_4096", "kind": "text", "w": 4096, "h": 4096, "font": "noto", "size": 12,
         "words": 6000, "typeset": False},
        # A vector document of the size of a detailed illustration.
        {"name": "document_900", "kind": "svg", "w": 900, "h": 900, "elements": 240, "gradient": True},
        # A whole canvas blurred.
        {"name": "blur_4096_r8", "kind": "blur", "w": 4096, "h": 4096, "radius": 8},
        # A drop shadow of a layer of odd size.
        {"name": "shadow_1921x1081", "kind": "shadow", "w": 1921, "h": 1081, "dx": 12.0, "dy": 12.0,
         "spread": 4, "blur": 16},
        # A layer composed: gradient fill, a rotated picture drawn on it, a
        # mask, opacity, and the layer blended onto its canvas.
        {"name": "layer_4096", "kind": "layer", "w": 4096, "h": 4096, "pic": 3000, "angle": 30.0,
         "zoom": 1.2, "paint": "radial", "mode": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: kinds as often as listed, sizes spread over their logarithm."""
    kind = rng.choice(["fill", "frame", "serve", "scene", "scene", "atlas", "text", "text", "svg", "blur",
                       "shadow", "layer"])
    w, h = _log_int(rng, 128, 4096), _log_int(rng, 128, 4096)
    if kind == "fill":
        return {"kind": kind, "w": w, "h": h, "points": _log_int(rng, 3, 400),
                "mode": rng.choice([0, 0, 1, 2, 5, 9])}
    if kind == "frame":
        return {"kind": kind, "w": min(w, 2560), "h": min(h, 1440), "ops": rng.randint(4, 40)}
    if kind == "serve":
        return {"kind": kind, "side": _log_int(rng, 256, 2048), "paths": _log_int(rng, 1, 100),
                "blur": rng.choice([0, 8])}
    if kind == "scene":
        return {"kind": kind, "w": w, "h": h, "paths": _log_int(rng, 4, 1500)}
    if kind == "atlas":
        return {"kind": kind, "w": _log_int(rng, 512, 8192), "glyphs": _log_int(rng, 100, 9000)}
    if kind == "text":
        size = rng.choice([9, 12, 14, 16, 24, 40])
        # as many words as about two thirds of the canvas hold
        words = max(4, int(w * h * 0.66 / (size * size * 4.5)))
        return {"kind": kind, "w": w, "h": h, "font": rng.choice(sorted(FONTS)), "size": size,
                "words": min(words, 6000), "typeset": bool(rng.getrandbits(1))}
    if kind == "svg":
        return {"kind": kind, "w": min(w, 2048), "h": min(h, 2048), "elements": _log_int(rng, 8, 1400),
                "gradient": bool(rng.getrandbits(1))}
    if kind == "blur":
        return {"kind": kind, "w": w, "h": h, "radius": _log_int(rng, 1, 40)}
    if kind == "shadow":
        return {"kind": kind, "w": w, "h": h, "dx": rng.choice([0.0, 3.0, 12.0, 2.5]),
                "dy": rng.choice([2.0, 12.0, -5.25]), "spread": rng.randint(0, 8), "blur": rng.randint(0, 24)}
    return {"kind": kind, "w": w, "h": h, "pic": _log_int(rng, 64, 3000), "angle": round(rng.uniform(0, 90), 2),
            "zoom": round(rng.uniform(0.3, 2.5), 3), "paint": rng.choice(["linear", "radial", "angular"]),
            "mode": rng.randint(0, 15)}


# ---- inputs ----

def _color(rng, lo=51):
    """A premultiplied colour of random alpha."""
    r, g, b = (int(v) for v in rng.integers(0, 256, 3))
    a = int(rng.integers(lo, 256))
    return tuple((c * a + 127) // 255 for c in (r, g, b)) + (a,)


def _loop(rng, w, h, side):
    """A closed path of 4..32 cubics inside a box of that side on the canvas."""
    side = min(side, w, h)
    n = int(rng.integers(4, 33))
    p = rng.uniform(0, side, (n, 6)) + np.tile([rng.uniform(0, w - side), rng.uniform(0, h - side)], 3)
    c = np.empty(3 + 7 * n + 1, np.float32)
    c[:3] = MOVE, p[-1, 4], p[-1, 5]
    body = c[3:-1].reshape(n, 7)
    body[:, 0] = CUBIC
    body[:, 1:] = p
    c[-1] = CLOSE
    return c


def _calls(rng, w, h, paths, max_side):
    """Fills in the 16 colour blend modes and both rules, three in ten also
    stroked, as (path, colour, keyword arguments, stroked)."""
    out = []
    for i in range(paths):
        c = _loop(rng, w, h, float(np.clip(rng.lognormal(math.log(64), 1.0), 4, max_side)))
        color = _color(rng)
        out.append((c, color, {"windingRule": int(rng.integers(0, 2)), "blendMode": i % 16}, False))
        if rng.random() < 0.3:
            kw = {"strokeWidth": float(rng.uniform(1, 8)), "lineCap": int(rng.integers(0, 3)),
                  "lineJoin": int(rng.integers(0, 3)), "blendMode": i % 16}
            if rng.random() < 0.1:
                kw["dashes"] = [float(v) for v in rng.uniform(2, 20, 2)]
            out.append((c, color, kw, True))
    return out


def _record(scene, calls):
    for c, color, kw, stroked in calls:
        (scene.strokePath if stroked else scene.fillPath)(c, color, **kw)


def _picture(seed, w, h, a8=False):
    """A random premultiplied image on the GPU: its bytes, and the image over them."""
    gen = torch.Generator("cuda").manual_seed(seed)
    if a8:
        t = torch.randint(0, 256, (h, w), generator=gen, dtype=torch.uint8, device="cuda")
    else:
        t = torch.randint(0, 256, (h, w, 4), generator=gen, dtype=torch.uint8, device="cuda")
        t = torch.minimum(t, t[..., 3:]).contiguous()
    torch.cuda.synchronize()
    return t, px.Image.view(t.data_ptr(), w, h, a8)


def _canvas(w, h, a8=False):
    t = torch.zeros((h, w) if a8 else (h, w, 4), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    return t, px.Image.view(t.data_ptr(), w, h, a8)


class _Pixels:
    """An image that the library allocated, as an array that keeps it alive."""

    def __init__(self, img):
        self.img = img
        self.__cuda_array_interface__ = {"shape": (img.height, img.width, 4), "typestr": "|u1", "version": 2,
                                         "data": (img.device_ptr(), False)}


def _pixels(img):
    return torch.as_tensor(_Pixels(img), device="cuda")


def _rotation(angle, zoom, tx, ty):
    c, s = zoom * math.cos(math.radians(angle)), zoom * math.sin(math.radians(angle))
    return np.array([c, s, 0, -s, c, 0, tx, ty, 1], np.float32)


def _gradient(rng, kind, w, h, mode):
    kinds = {"linear": px.PaintKind.LinearGradientPaint, "radial": px.PaintKind.RadialGradientPaint,
             "angular": px.PaintKind.AngularGradientPaint}
    at = [(w * float(rng.uniform(0.3, 0.7)), h * float(rng.uniform(0.3, 0.7)))]
    at.append((at[0][0] + 0.4 * w, at[0][1]))
    if kind != "linear":
        at.append((at[0][0], at[0][1] + 0.4 * h))
    stops = [px.ColorStop(tuple(float(v) for v in rng.uniform(0, 1, 4)), p) for p in (0.0, 0.4, 1.0)]
    return px.Paint(kinds[kind], blendMode=mode, opacity=0.8, gradientHandlePositions=at, gradientStops=stops)


def _rounded(w, h, x, y, r):
    p = px.Path()
    p.rounded_rect(x, y, w, h, r, r, r, r)
    return p.array()


def _frame_ops(rng, w, h, n):
    """(path, paint, keyword arguments, stroked): of every six, three panels, a
    blob, an outline and a gradient button."""
    ops = []
    for i in range(n):
        bw, bh = float(rng.uniform(0.05, 0.4)) * w, float(rng.uniform(0.05, 0.3)) * h
        x, y = float(rng.uniform(0, w - bw)), float(rng.uniform(0, h - bh))
        what = i % 6
        if what < 3:
            ops.append((_rounded(bw, bh, x, y, 0.2 * min(bw, bh)), _color(rng, 160), {}, False))
        elif what == 3:
            ops.append((_loop(rng, w, h, max(bw, bh)), _color(rng), {"windingRule": 1}, False))
        elif what == 4:
            kw = {"strokeWidth": float(rng.uniform(1, 6)), "lineJoin": 1}
            if i % 12 == 4:
                kw["dashes"] = [6.0, 3.0]
            ops.append((_rounded(bw, bh, x, y, 8.0), _color(rng), kw, True))
        else:
            ops.append((_rounded(bw, bh, x, y, 12.0), _gradient(rng, "linear", w, h, 0), {}, False))
    return ops


def _outline(rng):
    """A glyph-like outline in a unit box: 1..3 contours of quadratics."""
    parts = []
    for c in range(int(rng.integers(1, 4))):
        n = int(rng.integers(5, 40))
        scale = 0.48 if c == 0 else float(rng.uniform(0.1, 0.25))
        a = np.sort(rng.uniform(0, 2 * math.pi, n))
        am = (a + np.append(a[1:], a[0] + 2 * math.pi)) / 2
        if c:
            a, am = -a, -am
        r, rc = rng.uniform(0.6, 1.0, n) * scale, rng.uniform(0.5, 1.0, n) * scale
        on = 0.5 + np.stack([np.cos(a) * r, np.sin(a) * r], 1)
        ctl = 0.5 + np.stack([np.cos(am) * rc, np.sin(am) * rc], 1)
        q = np.concatenate([np.full((n, 1), QUAD), ctl, np.roll(on, -1, 0)], 1)
        parts += [[MOVE, *on[0]], q.reshape(-1), [CLOSE]]
    cmds = np.concatenate(parts).astype(np.float32)
    xs = np.zeros(len(cmds), np.int8)  # 1: an x, 2: a y, 0: a command kind
    i = 0
    while i < len(cmds):
        n = {MOVE: 2, QUAD: 4}.get(float(cmds[i]), 0)
        xs[i + 1:i + 1 + n:2], xs[i + 2:i + 1 + n:2] = 1, 2
        i += 1 + n
    return cmds, xs == 1, xs == 2


def _atlas_cells(aw, glyphs):
    """Cell positions and sizes, shelf by shelf, and the atlas's height: the
    same for every seed, as a program keeps its atlas's layout and size."""
    rng = np.random.default_rng(4)
    size = np.clip(rng.lognormal(math.log(32), 0.8, (glyphs, 2)), 8, 256).astype(int)
    cells, x, y, shelf = [], 0, 0, 0
    for w, h in size.tolist():
        if x + w + 1 > aw:
            x, y, shelf = 0, y + shelf + 1, 0
        cells.append((x, y, w, h))
        x, shelf = x + w + 1, max(shelf, h)
    return cells, y + shelf


_WORDS = ("she had come to the conclusion that you could tell a lot about person by their ears way they "
          "stuck out and size of earlobes give wonderful insights into of course scientifically prove any "
          "this but didn't matter her After all, that's what hunches are for 1984 Yes; (quite) so.").split()


def _text(rng, words):
    return " ".join(_WORDS[i] for i in rng.integers(0, len(_WORDS), words))


def _document(rng, w, h, elements, gradient):
    """An SVG document: curved shapes, some stroked, in nested groups."""
    hexc = lambda: "#%02x%02x%02x" % tuple(int(v) for v in rng.integers(0, 256, 3))  # noqa: E731
    out = ['<svg xmlns="http://www.w3.org/2000/svg" width="%d" height="%d" viewBox="0 0 %d %d">' % (w, h, w, h)]
    if gradient:
        out.append('<linearGradient id="bg" gradientUnits="userSpaceOnUse" x1="0" y1="0" x2="0" y2="%d">'
                   '<stop offset="0" stop-color="%s"/><stop offset="1" stop-color="%s"/></linearGradient>'
                   % (h, hexc(), hexc()))
        out.append('<rect x="0" y="0" width="%d" height="%d" fill="url(#bg)"/>' % (w, h))
    for i in range(elements):
        if i % 24 == 0:
            out.append('<g transform="translate(%.2f,%.2f)">' % tuple(rng.uniform(-0.05, 0.05, 2) * (w, h)))
        side = float(np.clip(rng.lognormal(math.log(0.06), 1.0), 0.01, 0.5)) * min(w, h)
        at = rng.uniform(0, 1, 2) * (w - side, h - side)
        style = 'fill="%s"' % hexc()
        if i % 3 == 1:
            style += ' stroke="%s" stroke-width="%.2f"' % (hexc(), rng.uniform(0.5, 4))
        if i % 5 == 2:
            style = 'fill="none" stroke="%s" stroke-width="%.2f" stroke-linecap="round"' % (hexc(),
                                                                                         rng.uniform(0.5, 3))
        if i % 8 == 7:
            out.append('<circle cx="%.2f" cy="%.2f" r="%.2f" %s/>' % (at[0], at[1], side / 2, style))
        else:
            n = int(rng.integers(3, 14))
            p = at + rng.uniform(0, side, (3 * n + 1, 2))
            d = "M%.2f,%.2f" % tuple(p[0])
            for k in range(n):
                d += "C" + " ".join("%.2f,%.2f" % tuple(q) for q in p[1 + 3 * k:4 + 3 * k])
            out.append('<path d="%sZ" %s/>' % (d, style))
        if i % 24 == 23 or i == elements - 1:
            out.append("</g>")
    return "\n".join(out + ["</svg>"])


# ---- the passes ----

def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "fill":
        w, h, n = case["w"], case["h"], case["points"]
        s["out"], s["img"] = _canvas(w, h)
        a = 2 * math.pi * np.arange(n) / n
        r = rng.uniform(0.3, 0.5, n)
        c = np.empty(3 * n + 1, np.float32)
        body = c[:-1].reshape(n, 3)
        body[:, 0] = LINE
        body[0, 0] = MOVE
        body[:, 1], body[:, 2] = w * (0.5 + r * np.cos(a)), h * (0.5 + r * np.sin(a))
        c[-1] = CLOSE
        s["path"], s["color"] = c, _color(rng, 255 if case["mode"] == 0 else 51)
    elif kind == "frame":
        s["out"], s["img"] = _canvas(case["w"], case["h"])
        s["ops"] = _frame_ops(rng, case["w"], case["h"], case["ops"])
    elif kind == "serve":
        side = case["side"]
        s["lanes"] = []
        for lane in range(1, px.lanes()):
            t, img = _canvas(side, side)
            s["lanes"].append((lane, t, img, px.Scene(), _calls(rng, side, side, case["paths"], side)))
    elif kind == "scene":
        s["out"], s["img"] = _canvas(case["w"], case["h"])
        s["scene"] = px.Scene()
        _record(s["scene"], _calls(rng, case["w"], case["h"], case["paths"], 2048))
    elif kind == "atlas":
        cells, ah = _atlas_cells(case["w"], case["glyphs"])
        s["out"], s["img"] = _canvas(case["w"], ah, a8=True)
        s["scene"] = px.Scene()
        glyphs = [_outline(rng) for _ in range(min(256, case["glyphs"]))]
        for i, (x, y, w, h) in enumerate(cells):
            c, xs, ys = glyphs[i % len(glyphs)]
            c = c.copy()
            c[xs] = c[xs] * w + x
            c[ys] = c[ys] * h + y
            s["scene"].fillPath(c, (255, 255, 255, 255))
    elif kind == "text":
        s["out"], s["img"] = _canvas(case["w"], case["h"])
        s["font"] = px.readFont(os.path.join(ROOT, "tests", "golden", "fonts", FONTS[case["font"]]))
        s["font"].size = case["size"]
        s["text"], s["bounds"] = _text(rng, case["words"]), (float(case["w"]), float(case["h"]))
        if not case["typeset"]:
            s["arrangement"] = px.typeset(s["font"], s["text"], bounds=s["bounds"])
    elif kind == "svg":
        s["svg"] = px.parseSvg(_document(rng, case["w"], case["h"], case["elements"], case["gradient"]))
    elif kind == "blur":
        s["keep"], s["src"] = _picture(seed, case["w"], case["h"])
        s["out"], s["img"] = _canvas(case["w"], case["h"])
    elif kind == "shadow":
        s["keep"], s["src"] = _picture(seed, case["w"], case["h"])
        s["color"] = _color(rng)
    else:
        w, h = case["w"], case["h"]
        s["keep"], s["pic"] = _picture(seed, case["pic"], case["pic"])
        s["keep2"], s["mask"] = _picture(seed + 1, w, h, a8=True)
        s["backdrop"] = _color(rng, 255)
        s["layer_px"], s["layer"] = _canvas(w, h)
        s["out"], s["img"] = _canvas(w, h)
        s["mat"] = _rotation(case["angle"], case["zoom"], 0.4 * w, -0.1 * h)
        s["path"] = _rounded(0.9 * w, 0.9 * h, 0.05 * w, 0.05 * h, 0.1 * min(w, h))
        s["paint"] = _gradient(rng, case["paint"], w, h, 0)
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "fill":
        s["img"].fillPath(s["path"], s["color"], blendMode=case["mode"])
    elif kind == "frame":
        img = s["img"]
        img.fill((255, 255, 255, 255))
        for c, paint, kw, stroked in s["ops"]:
            (img.strokePath if stroked else img.fillPath)(c, paint, **kw)
    elif kind == "serve":
        for lane, _, img, scene, calls in s["lanes"]:
            scene.clear()
            _record(scene, calls)
            img.fill((0, 0, 0, 0), lane=lane)
            scene.render(img, lane)
            if case["blur"]:
                img.blur(case["blur"], lane=lane)
        for lane, *_ in s["lanes"]:
            px.lane_synchronize(lane)
        return [t for _, t, *_ in s["lanes"]]
    elif kind == "scene":
        s["img"].fill((255, 255, 255, 255))
        s["scene"].render(s["img"])
    elif kind == "atlas":
        s["img"].fill((0, 0, 0, 0))
        s["scene"].render(s["img"])
    elif kind == "text":
        s["img"].fill((255, 255, 255, 255))
        if case["typeset"]:
            s["img"].fillText(s["font"], s["text"], bounds=s["bounds"])
        else:
            s["img"].fillText(s["arrangement"])
    elif kind == "svg":
        return _pixels(px.svg.newImage(s["svg"]))
    elif kind == "blur":
        s["img"].draw(s["src"], blendMode=px.BlendMode.Overwrite)
        s["img"].blur(case["radius"])
    elif kind == "shadow":
        return _pixels(s["src"].shadow((case["dx"], case["dy"]), case["spread"], case["blur"], s["color"]))
    else:
        layer, img = s["layer"], s["img"]
        img.fill(s["backdrop"])
        layer.fill((0, 0, 0, 0))
        layer.fillPath(s["path"], s["paint"])
        layer.draw(s["pic"], transform=s["mat"])
        layer.draw(s["mask"], blendMode=px.BlendMode.Mask)
        layer.applyOpacity(0.75)
        img.draw(layer, blendMode=case["mode"])
        return [s["layer_px"], s["out"]]
    return s["out"]


def work(case):
    """Each input read once and each output written once.  Paths are counted
    at the mean size of their command arrays; the operations are the taps of
    the blurs (a multiply and an add per tap, channel and direction), the only
    part whose number is fixed."""
    kind, flops = case["kind"], 0
    if kind == "fill":  # half the canvas is covered: read and written
        nbytes = 8 * 0.5 * case["w"] * case["h"] + 12 * case["points"]
    elif kind == "frame":
        nbytes = 4 * case["w"] * case["h"] + 200 * case["ops"]
    elif kind == "serve":
        px4 = 4 * (px.lanes() - 1) * case["side"] ** 2
        nbytes = px4 + 4 * (px.lanes() - 1) * case["paths"] * 520
        flops = 4 * px4 * (2 * case["blur"] + 1) if case["blur"] else 0
    elif kind == "scene":
        nbytes = 4 * case["w"] * case["h"] + case["paths"] * 520
    elif kind == "atlas":
        nbytes = case["w"] * _atlas_cells(case["w"], case["glyphs"])[1] + case["glyphs"] * 900
    elif kind == "text":  # about 5.6 glyphs a word, each placed (64 bytes)
        nbytes = 4 * case["w"] * case["h"] + case["words"] * 5.6 * 64
    elif kind == "svg":
        nbytes = 4 * case["w"] * case["h"] + case["elements"] * 230
    elif kind == "blur":
        nbytes = 8 * case["w"] * case["h"]
        flops = 16 * case["w"] * case["h"] * (2 * case["radius"] + 1)
    elif kind == "shadow":  # the blur runs on one channel: a shadow's colours are its alpha's
        nbytes = 8 * case["w"] * case["h"]
        flops = 4 * case["w"] * case["h"] * (2 * case["blur"] + 1)
    else:  # picture and mask read, layer and canvas written
        nbytes = 4 * case["pic"] ** 2 + 9 * case["w"] * case["h"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    return "exact"
