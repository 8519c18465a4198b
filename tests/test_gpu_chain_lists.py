"""GPU: the intersection work lists against the oracle, image bytes equal.

Curve counts around one block's 1024 and beyond 512 blocks (blocks then take several runs of
curves), and scenes whose curves lie almost all off the canvas, so that few cuts leave little
room for the blocks' counts.
"""
import numpy as np
import pytest

import pyoracle
import scanline
from scanline import VGContainer, rgba
from scanline.scene import KIND_GLYPHS

pytestmark = pytest.mark.gpu


def check(r, a, W, H):
    print("chain lists:", W, H, a.n_paths, a.n_curves, flush=True)
    ref = pyoracle.run(a, W, H, 8, srgb=True, ms=False, keep=False)
    r.setSamples(8)
    r.enableSRGBCorrection(True)
    r.setMultisampleOutput(False)
    r.resizeOutputBuffer(W, H)
    r.setInputTransform(np.eye(4, dtype=np.float32))
    r.dumpDebugData(False)
    r.addVg(a)
    r.rasterize()
    assert r.elementNumber() == ref.counts()
    np.testing.assert_array_equal(r.output(), ref.get("image").reshape(H, W, 4))


def triangles(W, H, n, shown, seed):
    """n triangles, 3 n curves; those from `shown` on lie below the canvas."""
    rng = np.random.default_rng(seed)
    vg = VGContainer(W, H)
    for k in range(n):
        vg.addPath(k & 1, rgba(*rng.integers(0, 256, 4)))
        x, y = rng.uniform(0, W), rng.uniform(0, H) + (0 if k < shown else 50 * H)
        vg.addPolygon([(x, y), (x + 7, y + 1), (x + 2, y + 8)])
    return vg.arrays()


@pytest.mark.parametrize("n", [341, 342, 683, 1366])
def test_curves_around_one_block(rasterizer, n):
    check(rasterizer, triangles(60, 50, n, n, n), 60, 50)


@pytest.mark.parametrize("shown", [0, 1, 3, 40])
def test_few_cuts_for_many_curves(rasterizer, shown):
    check(rasterizer, triangles(60, 50, 7000, shown, shown), 60, 50)


def test_more_curves_than_512_blocks_of_1024(rasterizer):
    a = scanline.generate(KIND_GLYPHS, 300, 300, 40000, 5)
    assert a.n_curves > 513 * 1024
    check(rasterizer, a, 300, 300)
