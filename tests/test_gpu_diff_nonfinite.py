"""GPU: crossings without a position in the differentiable mode.

A control point whose x is not finite, its y being finite, gives crossings at NaN.  They end
their row's order and lie at the canvas's right edge, so a row's coverage stays what fills
its pixels once: in [0, 1], the same bits for every run, and untouched where the path's row
has finite crossings only.
"""
import numpy as np
import pytest
import torch

import pyoracle
import scanline
from scanline import diff

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def scene(W, H):
    """Three stacked black boxes; the middle one's sides are the cases'."""
    vg = scanline.VGContainer()
    for k, (y0, y1) in enumerate(((1, 4), (5, 9), (10, 13))):
        vg.addPath(k & 1, scanline.rgba(0, 0, 0, 255))
        vg.addPolygon([(10.25, y0), (W - 7.5, y0), (W - 7.5, y1), (10.25, y1)])
        # a quadratic bump beside it, whose bend point a case may take out
        vg.addQuadratic((10.25, y1), (2.0, 0.5 * (y0 + y1)), (10.25, y0))
        vg.addLinear((10.25, y0), (10.25, y1))
    return vg.arrays()


@pytest.mark.parametrize("W", [40, 600])
@pytest.mark.parametrize("slots,x", [
    ((2, 3), NAN), ((2, 3), INF), ((2, 3), -INF),       # the right side
    ((6, 7), NAN), ((6, 7), -NAN), ((6, 7), INF),       # the left side
    ((2,), NAN), ((9,), NAN), ((9,), -INF), ((2, 3, 6, 7, 9), NAN)])
def test_coverage_stays_in_its_range(slots, x, W):
    H, rows = 14, 8
    print("diff nonfinite:", slots, x, W, flush=True)
    a = scene(W, H)
    first = a.curve_vertex_pos[np.flatnonzero(a.curve_path_id == 1)[0]]
    pts = a.vertex.copy()
    for s in slots:
        pts[first + s, 0] = x
    r = diff.DiffRenderer(a, W, H, samples=rows)
    try:
        p = torch.tensor(pts, device="cuda")
        cov = 1.0 - r.forward_raw(p, r.colors0, keep=False)[:, :, 0].cpu().numpy()
        again = 1.0 - r.forward_raw(p, r.colors0, keep=False)[:, :, 0].cpu().numpy()
        assert np.array_equal(cov, again)
        # coverages are sums of exact parts: their rounding to float and 1 - (1 - c) leave 2^-24
        assert cov.min() >= -2.0 ** -23 and cov.max() <= 1.0 + 2.0 ** -23
        ref, _, _, _ = pyoracle.diff_run(a, W, H, samples=rows, double=False)
        whole = [y for y in range(H) if not 5 <= y < 9]
        np.testing.assert_allclose(cov[whole], 1.0 - ref[whole][:, :, 0], rtol=0, atol=1e-5)
    finally:
        r.close()
