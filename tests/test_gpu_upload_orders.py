"""GPU: scenes whose curves' vertices follow one another, and the same scenes with the
vertices in another order or with unused ones between, give the same image bytes; shared
vertices are refused in both.
"""
import numpy as np
import pytest

import scanline
from scanline.scene import KIND_GLYPHS, KIND_MIXED, SceneArrays

pytestmark = pytest.mark.gpu


def image(r, a, W, H):
    print("upload:", a.n_paths, a.n_curves, a.n_vertices, flush=True)
    r.setSamples(8)
    r.enableSRGBCorrection(True)
    r.setMultisampleOutput(False)
    r.resizeOutputBuffer(W, H)
    r.setInputTransform(np.eye(4, dtype=np.float32))
    r.dumpDebugData(False)
    r.addVg(a)
    r.rasterize()
    return r.output()


def moved(a, order, gap):
    """The scene with its curves' vertex runs laid out in `order`, `gap` unused between."""
    nv = (a.curve_type & 7).astype(np.int64)
    pos = np.zeros(a.n_curves, np.int64)
    pos[order] = np.concatenate([[0], np.cumsum(nv[order] + gap)[:-1]])
    v = np.full((int((nv + gap).sum()), 2), 3.0, np.float32)
    src = a.vertex.reshape(-1, 2)
    for k in range(4):
        m = nv > k
        v[pos[m] + k] = src[a.curve_vertex_pos[m] + k]
    return SceneArrays(v, pos.astype(np.uint32), a.curve_type, a.curve_path_id, a.curve_arc_w, a.fill_rule, a.fill_color)


@pytest.mark.parametrize("kind,paths", [(KIND_MIXED, 40), (KIND_GLYPHS, 1300)])  # below and above 65536 curves
def test_vertex_orders(rasterizer, kind, paths):
    a = scanline.generate(kind, 200, 150, paths, 3)
    ref = image(rasterizer, a, 200, 150)
    n = a.n_curves
    order = np.arange(n)
    swapped = order.copy()
    swapped[[n // 2, n // 2 + 1]] = swapped[[n // 2 + 1, n // 2]]
    for o, gap in [(order, 2), (order[::-1], 0), (swapped, 0), (np.random.default_rng(1).permutation(n), 1)]:
        np.testing.assert_array_equal(image(rasterizer, moved(a, o, gap), 200, 150), ref)


@pytest.mark.parametrize("at", [0, 1, 19])
def test_shared_vertices_are_refused(rasterizer, at):
    a = scanline.generate(KIND_MIXED, 60, 60, 5, 4)
    pos = a.curve_vertex_pos.copy()
    pos[at + 1] = pos[at]
    b = SceneArrays(a.vertex, pos, a.curve_type, a.curve_path_id, a.curve_arc_w, a.fill_rule, a.fill_color)
    with pytest.raises(scanline.ScanlineError, match="vertex %d belongs to two curves" % pos[at]):
        rasterizer.addVg(b)
