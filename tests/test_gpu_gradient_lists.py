"""GPU: gradient paints in the compositors' bucket lists, against the oracle.

A tile's buckets are listed up to 64 at a time and blended in groups of a few; gradients and
solid paints alternate.  Path counts around one and two lists and around the groups, spans
that reach past the tile on either side (the covering item's ends lie in the neighbouring
records or at the bucket's extent), separate bars within a tile, one and several tiles.
"""
import numpy as np
import pytest

import pyoracle
from scanline import VGContainer, rgba
from scanline.gradient import GradientTextures
from scanline.scene import SceneArrays

pytestmark = pytest.mark.gpu

STOPS = [(0.0, 0.1, 0.9, 0.3, 0.5), (0.4, 1.0, 0.2, 0.1, 0.9), (1.0, 0.0, 0.3, 1.0, 0.7)]


def scene(W, H, n, srgb):
    rng = np.random.default_rng(W + n)
    vg = VGContainer(W, H)
    g = GradientTextures(srgb=srgb)
    for k in range(n):
        vg.addPath(k & 1, rgba(*rng.integers(0, 256, 3), 255 if k % 5 == 0 else 140))
        if k % 3 == 2:  # bars with gaps
            for x in np.arange(3.0 + k % 7, W, 23.0):
                vg.addPolygon([(x, 0.4), (x + 9.5, 0.4), (x + 8.0, H - 0.6), (x, H - 0.6)])
        else:
            x0, x1 = np.sort(rng.uniform(-20, W + 20, 2))
            vg.addPolygon([(x0, 0.2), (x1, 0.7), (x1 + 2.5, H - 0.5), (x0 - 1.0, H - 0.1)])
        if k % 4 == 3:
            g.add_solid()
        else:
            g.add("linear" if k & 1 else "radial", 0.2 * W, 3.0, 0.8 * W, 6.0, 0.4 * W, STOPS, 0.8,
                  [1.0, 0.1, 2.0, 0.0, 0.9, 1.0])
    a = vg.arrays()
    fill = a.fill_color.copy()
    painted = np.arange(n) % 4 != 3
    fill[painted] = np.flatnonzero(painted) + 1
    ramp, table = g.textures()
    return SceneArrays(a.vertex, a.curve_vertex_pos, a.curve_type, a.curve_path_id, a.curve_arc_w, a.fill_rule, fill,
                       ramp, table)


@pytest.mark.parametrize("spp", [8, 16, 32])
@pytest.mark.parametrize("ms,srgb", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("W,n", [(50, 1), (64, 2), (130, 5), (200, 63), (70, 64), (131, 67), (65, 130)])
def test_lists_of_gradients(rasterizer, W, n, ms, srgb, spp):
    H = 9
    print("gradient lists:", W, n, "ms" if ms else "cov", srgb, spp, flush=True)
    a = scene(W, H, n, srgb)
    ref = pyoracle.run(a, W, H, spp, srgb=srgb, ms=ms, keep=False)
    r = rasterizer
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
