"""GPU: coverages of thin slivers in the differentiable mode.

Left of x = 1/4 a float position is finer than the 2^-25 of a sample row that a row's sums
are kept in; the first column keeps what lies below.  The coverage of a bar of width w in it
is read off the colour gradient -- the sum of image gradient times coverage, with a gradient
large enough for the sum to lie near 1 -- and compared with the float oracle's, which takes
the same crossings.

Tolerance: the oracle sums 16 quotients of a difference, each rounded, 16 * 2^-24; the kernels
keep 2^-56 of a row, 2^-24 of the narrowest bar, round twice, and sum four rows; together
below 2e-6 of the value.
"""
import numpy as np
import pytest
import torch

import pyoracle
import scanline
from scanline import diff

pytestmark = pytest.mark.gpu

BARS = [(1e-3, 1e-6), (2e-4, 3e-8), (1e-6, 1e-9), (0.1, 1.5e-8), (3e-8, 2e-10), (-5.0, 5.0 + 1e-9), (0.24, 1e-7),
        (0.3, 1e-6), (5.0, 2e-6), (0.05, 1.9)]


@pytest.mark.parametrize("rows", [16, 64, 3])
@pytest.mark.parametrize("x0,w", BARS)
def test_bar(x0, w, rows):
    W, H = 8, 4
    x1 = np.float32(1e-9) if x0 < 0 else np.float32(x0 + w)
    x0 = np.float32(x0)
    assert x1 > x0
    vg = scanline.VGContainer()
    vg.addPath(0, scanline.rgba(0, 0, 0, 255))
    vg.addPolygon([(x0, -1.0), (x1, -1.0), (x1, H + 1.0), (x0, H + 1.0)])
    a = vg.arrays()
    r = diff.DiffRenderer(a, W, H, samples=rows)
    try:
        scale = 2.0 ** -np.floor(np.log2(max(float(x1) - max(float(x0), 0.0), 1e-12)))
        g = np.zeros((H, W, 4), np.float32)
        g[:, :, 0] = scale
        r.forward_raw(r.points0, r.colors0)
        _, gc = r.backward_raw(torch.tensor(g, device="cuda"))
        _, _, rc, _ = pyoracle.diff_run(a, W, H, grad_image=g, samples=rows, double=False)
        print("sliver", x0, x1, rows, gc[0, 0].item(), rc[0, 0], flush=True)
        assert rc[0, 0] > 0
        assert abs(gc[0, 0].item() - rc[0, 0]) <= 2e-6 * (rows / 16 if rows > 16 else 1) * rc[0, 0]
    finally:
        r.close()
