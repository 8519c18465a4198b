"""GPU: intersections of frames that solve cubic chains with several lanes each.

The rule is by the frame's cuts (2^18, 2^21, 5 * 2^20, ...) and the piece's (24, 64, 128).
Scenes on each side of the first three limits are compared with the oracle, every intersection bit for
bit; so are control points far outside the canvas, whose coordinates carry so much rounding
that the signs along a piece change more than once (the walk through the sign bits), curves
with coincident and nearly coincident control points, one-pixel-wide canvases, and counts of
chains that leave rows and waves of the last group empty.  The image follows from the
intersections and is compared too.
"""
import numpy as np
import pytest

import pyoracle
import scanline
from scanline.scene import SceneArrays

pytestmark = pytest.mark.gpu


def check(r, a, W, H, spp=8, limits=None):
    print("wide chains:", W, H, a.n_curves, flush=True)
    r.setSamples(spp)
    r.enableSRGBCorrection(True)
    r.setMultisampleOutput(False)
    r.resizeOutputBuffer(W, H)
    r.setInputTransform(np.eye(4, dtype=np.float32))
    r.dumpDebugData(True)
    r.addVg(a)
    r.rasterize()
    ref = pyoracle.run(a, W, H, spp, srgb=True, ms=False)
    F = r.elementNumber()["curve_fragment"]
    if limits:
        assert limits[0] < F <= limits[1], F
    np.testing.assert_array_equal(r.dump("ts"), ref.get("ts"))
    np.testing.assert_array_equal(r.output(), ref.get("image").reshape(H, W, 4))
    r.dumpDebugData(False)


@pytest.mark.parametrize("W,H,paths,limits", [
    (640, 480, 40, (0, 1 << 18)), (640, 480, 150, (1 << 18, 1 << 21)), (1400, 1100, 420, (1 << 21, 5 << 20)),
    (2048, 2048, 900, (5 << 20, 1 << 24)),
    (64, 64, 1, (0, 1 << 18)), (50, 333, 3, (0, 1 << 18)), (1, 300, 5, (0, 1 << 18)), (300, 1, 5, (0, 1 << 18))])
def test_frames_on_each_side_of_the_limits(rasterizer, W, H, paths, limits):
    check(rasterizer, scanline.generate(scanline.scene.KIND_CUBIC_CHAINS, W, H, paths, 0x71DE + W), W, H, limits=limits)


@pytest.mark.parametrize("scale", [50.0, 3e3, 2e5])
def test_coordinates_with_much_rounding(rasterizer, scale):
    W = H = 512
    a = scanline.generate(scanline.scene.KIND_CUBIC_CHAINS, W, H, 25, 0x0DD + int(scale))
    a.vertex[:] = (a.vertex - np.float32(256)) * np.float32(scale) + np.float32(256)
    check(rasterizer, a, W, H)


def test_degenerate_cubics(rasterizer):
    rng = np.random.default_rng(9)
    v = []
    for k in range(40):
        p = rng.uniform(0, 400, 2)
        q = rng.uniform(0, 400, 2)
        e = 10.0 ** -rng.integers(1, 7)
        v += [p, p + e, q - e, q]                       # handles next to the ends
        v += [q, q, p + rng.uniform(-3, 3, 2), p] if k % 3 else [q, (p + q) / 2, (p + q) / 2, p]
    v = np.array(v, np.float32)
    # closed two-curve outlines: the second ends where the first starts
    v.reshape(40, 8, 2)[:, 4] = v.reshape(40, 8, 2)[:, 3]
    v.reshape(40, 8, 2)[:, 7] = v.reshape(40, 8, 2)[:, 0]
    n = 80
    a = SceneArrays(v, 4 * np.arange(n), np.full(n, 4), np.repeat(np.arange(40), 2), np.full(n, -1.0),
                    np.arange(40) & 1, np.full(40, 0xC04080FF))
    check(rasterizer, a, 400, 400, spp=16)
