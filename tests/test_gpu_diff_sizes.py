"""GPU: the differentiable mode at the sizes where its kernels change course: canvas widths
around one pass of the coverage kernel (512 columns), rows with more crossings than its LDS
stage holds, sample-row counts that are no power of two and the largest, path counts around
the adjoint's block of 256, one-pixel canvases.

Tolerances.  The float oracle takes the same crossings; it sums a pixel's intervals in
float, each addition within 2^-24 of a coverage of at most 1.  The longest sums here hold
about 700 intervals, 4.2e-5, and compositing carries a coverage error with a weight of at
most 1 per path: 1e-4 bounds the image.  Gradients: 1e-4 of their norm, as in
test_gpu_diff.py.
"""
import numpy as np
import pytest
import torch

import pyoracle
import scanline
from scanline import diff

pytestmark = pytest.mark.gpu

CASES = [  # kind, width, height, rows, paths, segments
    ("cubics", 511, 9, 16, 6, 5), ("cubics", 512, 8, 16, 6, 5), ("mixed", 513, 9, 16, 12, 7),
    ("cubics", 1030, 5, 3, 5, 6), ("mixed", 33, 17, 64, 9, 6), ("cubics", 40, 6, 4, 3, 120),
    ("cubics", 16, 8, 4, 256, 4), ("mixed", 16, 8, 5, 257, 4), ("cubics", 1, 1, 16, 3, 4), ("mixed", 65, 1, 1, 8, 3),
]


@pytest.mark.parametrize("kind,W,H,rows,paths,segs", CASES)
def test_image_and_gradients(kind, W, H, rows, paths, segs):
    print("diff sizes:", kind, W, H, rows, paths, segs, flush=True)
    k = scanline.scene.KIND_CUBIC_CHAINS if kind == "cubics" else scanline.scene.KIND_MIXED
    scene = scanline.generate(k, W, H, paths, 0xD1FF + W, segs, segs)
    r = diff.DiffRenderer(scene, W, H, samples=rows)
    try:
        pts = r.points0.clone().requires_grad_(True)
        col = (r.colors0 * 0.9 + 0.05).clone().requires_grad_(True)
        img = r.render(pts, col)
        g = torch.tensor(np.random.default_rng(W).standard_normal((H, W, 4)).astype(np.float32), device="cuda")
        gp, gc = torch.autograd.grad(img, (pts, col), g)
        gp2, gc2 = torch.autograd.grad(r.render(pts, col), (pts, col), g)
        assert torch.equal(gp, gp2) and torch.equal(gc, gc2)
        ref, rp, rc, n = pyoracle.diff_run(scene, W, H, colors=col.detach().cpu().numpy(), grad_image=g.cpu().numpy(),
                                           samples=rows, double=False)
        assert r.crossings() == n
        np.testing.assert_allclose(img.detach().cpu().numpy(), ref, rtol=0, atol=1e-4)
        for a, b in ((gp, rp), (gc, rc)):
            a = a.cpu().numpy().astype(np.float64)
            assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b) + 1e-6
    finally:
        r.close()
