"""GPU: a view that shows little of a large scene costs no more than one that shows more.

The passes over a scene's curves are shared by as many blocks for a handful of cuts as for
thousands.  The intersection stage of 560000 curves with some 100 cuts in view is compared
with that of the same curves with some 20000: the best of several frames each, and a factor of
two for the clock's noise (one block for all curves took 30 times as long).
"""
import numpy as np
import pytest

import scanline
from scanline.scene import KIND_GLYPHS

pytestmark = pytest.mark.gpu


def stage(r, shift):
    m = np.eye(4, dtype=np.float32)
    m[3, 0] = m[3, 1] = shift
    r.setInputTransform(m)
    ms = []
    for _ in range(6):
        r.rasterize()
        ms.append(r.stepTiming()["intersect"])
    return min(ms), r.elementNumber()["curve_fragment"]


def test_few_cuts_of_many_curves(rasterizer):
    r, W, H = rasterizer, 600, 600
    r.setSamples(8)
    r.setMultisampleOutput(False)
    r.dumpDebugData(False)
    r.resizeOutputBuffer(W, H)
    a = scanline.generate(KIND_GLYPHS, W, H, 42000, 5)
    assert a.n_curves > 512 * 1024
    # moved by (t, t) a path is in view while the larger of its lowest x and y is below 600 - t
    first = a.curve_vertex_pos[np.searchsorted(a.curve_path_id, np.arange(a.n_paths))]
    low = np.sort(np.minimum.reduceat(a.vertex, first).max(1))
    r.addVg(a)
    r.enableStepTiming(True)
    try:
        many, nmany = stage(r, W - 0.5 * (low[299] + low[300]))
        few, nfew = stage(r, W - 0.5 * (low[0] + low[1]))
    finally:
        r.enableStepTiming(False)
        r.setInputTransform(np.eye(4, dtype=np.float32))
    print("few cuts:", nfew, "in %.3f ms," % few, nmany, "in %.3f ms" % many, flush=True)
    assert 0 < nfew < 202 < 8000 < nmany
    assert few <= 2.0 * many
