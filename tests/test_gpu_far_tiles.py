"""GPU: spans that run on past the 63rd tile of a bucket of many fragments.

A bucket's tile bitmaps end at its 63rd tile; from there on a column finds its span through
the flag that the resolve sets in the record before it.  Rows of packed narrow bars, as many as
fall to each of the resolve's passes (up to 64, 65..128, 129..1024, more than 1024
fragments), are followed by bars of 300 to 900 pixels beyond that tile, so that the
record that gets the flag lies in the same chunk, in an earlier one, and before any.  Images
are the oracle's, byte for byte.
"""
import numpy as np
import pytest

import pyoracle
from scanline import VGContainer, rgba

pytestmark = pytest.mark.gpu

W, H = 9000, 5


def bars(vg, xs, rule=0, color=(30, 90, 200, 170)):
    vg.addPath(rule, rgba(*color))
    for x0, x1 in xs:
        vg.addPolygon([(x0, 0.5), (x1, 0.5), (x1, 4.5), (x0, 4.5)])


def scene(narrow, seed):
    rng = np.random.default_rng(seed)
    vg = VGContainer(W, H)
    step = 3.0 if narrow < 1000 else 2.25
    first = [(4.0 + step * k, 4.0 + step * k + 1.5) for k in range(narrow)]
    far, x = [], max(64 * 64.0 + 20, first[-1][1] + 70) if first else 10.0
    while x < W - 40:
        w = float(rng.choice([300.0, 520.5, 900.0]))
        far.append((x, x + w))
        x += w + float(rng.choice([3.0, 66.0, 129.5]))
    bars(vg, first + far)
    # one span from the packed bars to the end, and bars packed at the far end as well
    bars(vg, first + [(first[-1][1] + 9.0, W - 30.0)] if first else far, color=(200, 60, 30, 120))
    bars(vg, first[: narrow // 2] + [(700.0, 8000.0)] + [(8100.0 + step * k, 8101.5 + step * k) for k in range(narrow // 2)
                                                       if 8101.5 + step * k < W], rule=1, color=(20, 200, 90, 255))
    return vg.arrays()


@pytest.mark.parametrize("ms,spp", [(False, 8), (True, 8), (True, 32)])
@pytest.mark.parametrize("narrow", [2, 20, 40, 200, 700])
def test_spans_beyond_the_bitmaps(rasterizer, narrow, ms, spp):
    a = scene(narrow, narrow)
    print("far tiles:", narrow, a.n_curves, ms, spp, flush=True)
    ref = pyoracle.run(a, W, H, spp, srgb=True, ms=ms, keep=False)
    r = rasterizer
    r.setSamples(spp)
    r.enableSRGBCorrection(True)
    r.setMultisampleOutput(ms)
    r.resizeOutputBuffer(W, H)
    r.setInputTransform(np.eye(4, dtype=np.float32))
    r.dumpDebugData(False)
    r.addVg(a)
    r.rasterize()
    assert r.elementNumber() == ref.counts()
    np.testing.assert_array_equal(r.output(), ref.get("image").reshape(H, W, 4))
