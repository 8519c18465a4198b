"""GPU: scenes whose vertex runs are out of order, or apart, against the oracle.

A scene whose curves' vertices follow one another is uploaded without claiming each vertex;
others claim them.  Both uploads render the oracle's image, byte for byte, below and above the
curve count from which host threads share the work.
"""
import numpy as np
import pytest

import pyoracle
import scanline
from scanline.scene import KIND_GLYPHS, KIND_MIXED, SceneArrays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,paths", [(KIND_MIXED, 40), (KIND_GLYPHS, 1300)])
@pytest.mark.parametrize("layout", ["as built", "gaps", "reversed", "shuffled"])
def test_layouts(rasterizer, layout, kind, paths):
    W, H = 200, 150
    a = scanline.generate(kind, W, H, paths, 7)
    n = a.n_curves
    assert (n >= 65536) == (paths == 1300)
    nv = (a.curve_type & 7).astype(np.int64)
    order = np.arange(n)
    if layout == "reversed":
        order = order[::-1]
    if layout == "shuffled":
        order = np.random.default_rng(2).permutation(n)
    gap = 2 if layout == "gaps" else 0
    pos = np.zeros(n, np.int64)
    pos[order] = np.concatenate([[0], np.cumsum(nv[order] + gap)[:-1]])
    v = np.full((int((nv + gap).sum()), 2), -3.0, np.float32)
    for k in range(4):
        m = nv > k
        v[pos[m] + k] = a.vertex[a.curve_vertex_pos[m] + k]
    b = SceneArrays(v, pos, a.curve_type, a.curve_path_id, a.curve_arc_w, a.fill_rule, a.fill_color)
    print("upload layout:", layout, n, b.n_vertices, flush=True)
    ref = pyoracle.run(a, W, H, 16, srgb=True, ms=False, keep=False)
    r = rasterizer
    r.setSamples(16)
    r.enableSRGBCorrection(True)
    r.setMultisampleOutput(False)
    r.resizeOutputBuffer(W, H)
    r.setInputTransform(np.eye(4, dtype=np.float32))
    r.dumpDebugData(False)
    r.addVg(b)
    r.rasterize()
    got = dict(r.elementNumber(), vertex=a.n_vertices)
    assert got == ref.counts()
    np.testing.assert_array_equal(r.output(), ref.get("image").reshape(H, W, 4))
