"""GPU: the compositors' tile records against the oracle, image bytes equal.

Rectangles with edges on, one pixel beside and halfway across tile boundaries (64 pixels),
spans that start or end off the canvas, canvas widths around one and two tiles, buckets
wider than the 63 tiles their bitmaps hold (canvases of up to 9000 pixels), zigzags whose
rows hold from a few to more than a thousand crossings (every size class of the resolve,
each with runs across tile boundaries), opaque paints over translucent ones and the
reverse, and gradients along spans that start and end in other tiles.
"""
import numpy as np
import pytest

import pyoracle
import scanline
from scanline import VGContainer, rgba
from scanline.gradient import GradientTextures
from scanline.scene import SceneArrays

pytestmark = pytest.mark.gpu


def check(r, a, W, H, spp=16, ms=False, srgb=True):
    print("tile records:", W, H, a.n_paths, "ms" if ms else "cov", flush=True)
    ref = pyoracle.run(a, W, H, spp, srgb=srgb, ms=ms, keep=False)
    r.setSamples(spp)
    r.enableSRGBCorrection(srgb)
    r.setMultisampleOutput(ms)
    r.resizeOutputBuffer(W, H)
    r.setInputTransform(np.eye(4, dtype=np.float32))
    r.dumpDebugData(False)
    r.addVg(a)
    r.rasterize()
    assert r.elementNumber() == ref.counts()
    np.testing.assert_array_equal(r.output(), ref.get("image").reshape(H, W, 4))


def rects(W, H, boxes, alpha=(255, 120)):
    vg = VGContainer(W, H)
    for k, (x0, x1) in enumerate(boxes):
        vg.addPath(k & 1, rgba(40 + 50 * k % 200, 90 + 31 * k % 150, 200 - 17 * k % 180, alpha[k % len(alpha)]))
        y0, y1 = 0.3 + 0.1 * (k % 5), H - 0.7 - 0.2 * (k % 3)
        vg.addPolygon([(x0, y0), (x1, y0), (x1, y1), (x0, y1)])
    return vg.arrays()


@pytest.mark.parametrize("W", [1, 2, 62, 63, 64, 65, 66, 127, 128, 129, 200])
@pytest.mark.parametrize("ms", [False, True])
def test_rectangles_at_tile_edges(rasterizer, W, ms):
    e = [-70.0, -2.0, 0.0, 1.0, 62.0, 63.0, 63.5, 64.0, 65.0, 66.0, 126.5, 128.0, 130.0, W - 1.0, W + 0.0, W + 90.0]
    boxes = [(a, b) for i, a in enumerate(e) for b in e[i + 1:] if b > a][::3]
    check(rasterizer, rects(W, 7, boxes), W, 7, ms=ms)


@pytest.mark.parametrize("W", [4033, 4096, 4160, 9000])
@pytest.mark.parametrize("ms", [False, True])
def test_buckets_wider_than_their_bitmaps(rasterizer, W, ms):
    rng = np.random.default_rng(W)
    boxes = [(-5.0, W + 5.0), (0.0, 4032.0), (0.0, 4033.0), (1.0, 4031.5), (70.0, W - 3.0), (4000.0, W - 1.5)]
    boxes += [tuple(sorted(rng.uniform(-10, W + 10, 2))) for _ in range(12)]
    a = rects(W, 5, boxes, alpha=(200, 255, 90))
    # one path of many separate bars: records, gaps and spans over the whole width
    vg = VGContainer.from_arrays(a)
    vg.addPath(0, rgba(250, 30, 30, 140))
    x = 3.0
    while x < W - 4:
        w = float(rng.choice([1.0, 30.0, 64.0, 200.0, 900.0]))
        vg.addPolygon([(x, 0.5), (x + w, 0.5), (x + w, 4.5), (x, 4.5)])
        x += w + float(rng.choice([2.0, 64.0, 130.0, 700.0]))
    check(rasterizer, vg.arrays(), W, 5, ms=ms)


@pytest.mark.parametrize("teeth", [3, 7, 8, 15, 16, 17, 31, 33, 63, 65, 130, 260, 600])
def test_zigzag_rows(rasterizer, teeth):
    W, H = 2100, 6
    vg = VGContainer(W, H)
    for k, (off, al) in enumerate([(0.0, 255), (13.3, 130)]):
        vg.addPath(k, rgba(30, 160 - 60 * k, 220, al))
        step = (W - 60.0) / teeth
        pts = [(20.0 + off, -3.0)]
        for i in range(teeth):
            pts += [(20.0 + off + step * (i + 0.25), 9.0), (20.0 + off + step * (i + 1), -2.0)]
        vg.addPolygon(pts)
    check(rasterizer, vg.arrays(), W, H, spp=32)


def test_deep_stacks_of_opaque_and_translucent_paints(rasterizer):
    rng = np.random.default_rng(3)
    vg = VGContainer(150, 40)
    for k in range(300):  # more than one list of 64 in every tile
        x0, x1 = np.sort(rng.uniform(-10, 160, 2))
        y0, y1 = np.sort(rng.uniform(-5, 45, 2))
        vg.addPath(k & 1, rgba(*rng.integers(0, 256, 3), 255 if rng.random() < 0.3 else int(rng.integers(1, 255))))
        vg.addPolygon([(x0, y0), (x1, y0 + 3), (x1 - 2, y1), (x0, y1)])
    for ms in (False, True):
        for srgb in (False, True):
            check(rasterizer, vg.arrays(), 150, 40, spp=8, ms=ms, srgb=srgb)


@pytest.mark.parametrize("W", [130, 700, 4600])
@pytest.mark.parametrize("ms", [False, True])
def test_gradients_along_spans(rasterizer, W, ms):
    a = rects(W, 9, [(0.5, W - 0.5), (-20.0, W + 20.0), (10.0, W - 30.25), (64.0, W - 2.0), (3.0, 61.0)], alpha=(255,))
    g = GradientTextures(srgb=True)
    fill = a.fill_color.copy()
    stops = [(0.0, 0.1, 0.9, 0.3, 0.5), (0.4, 1.0, 0.2, 0.1, 0.9), (1.0, 0.0, 0.3, 1.0, 0.7)]
    for p in range(a.n_paths):
        if p == 2:
            g.add_solid()
            continue
        g.add("linear" if p & 1 else "radial", 0.2 * W, 3.0, 0.8 * W, 6.0, 0.4 * W, stops, 0.8, [1.0, 0.1, 2.0, 0.0, 0.9, 1.0])
        fill[p] = p + 1
    ramp, table = g.textures()
    b = SceneArrays(a.vertex, a.curve_vertex_pos, a.curve_type, a.curve_path_id, a.curve_arc_w, a.fill_rule, fill, ramp, table)
    check(rasterizer, b, W, 9, spp=16, ms=ms)
