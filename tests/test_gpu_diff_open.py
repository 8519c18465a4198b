"""GPU: contours that do not close, in the differentiable mode.

The vertex slots of a scene are per segment, so points optimised slot by slot leave the
shared ends of their contours, and a row's windings need not return to zero.  The model
fills between a row's crossings only: nothing lies to the right of the last one, whatever
winding is left, in the oracle's sums and in the kernels'.

Tolerances as in test_gpu_diff_sizes.py: the float oracle takes the same crossings and sums a
pixel's intervals in float, at most about 700 of them, so 1e-4 bounds the image, and the
gradients agree within 1e-4 of their norm.
"""
import numpy as np
import pytest
import torch

import pyoracle
import scanline
from scanline import diff

pytestmark = pytest.mark.gpu

CASES = [  # kind, width, height, rows, paths, segments, moved by
    ("cubics", 96, 64, 16, 12, 6, 0.05), ("cubics", 96, 64, 16, 12, 6, 0.5), ("mixed", 96, 64, 16, 12, 7, 0.5),
    ("mixed", 700, 9, 8, 9, 6, 2.0),        # two passes over a row's columns
    ("cubics", 40, 6, 4, 3, 120, 0.5),      # rows beyond the crossings staged at once
]


@pytest.mark.parametrize("rule", [0, 1])
@pytest.mark.parametrize("kind,W,H,rows,paths,segs,by", CASES)
def test_points_moved_slot_by_slot(kind, W, H, rows, paths, segs, by, rule):
    print("diff open:", kind, W, H, rows, paths, segs, by, rule, flush=True)
    k = scanline.scene.KIND_CUBIC_CHAINS if kind == "cubics" else scanline.scene.KIND_MIXED
    scene = scanline.generate(k, W, H, paths, 0x09E2 + W, segs, segs)
    scene.fill_rule[:] = rule
    rng = np.random.default_rng(W + segs)
    moved = (scene.vertex + rng.uniform(-by, by, scene.vertex.shape)).astype(np.float32)
    g = rng.standard_normal((H, W, 4)).astype(np.float32)
    r = diff.DiffRenderer(scene, W, H, samples=rows)
    try:
        pts = torch.tensor(moved, device="cuda", requires_grad=True)
        col = (r.colors0 * 0.9 + 0.05).clone().requires_grad_(True)
        img = r.render(pts, col)
        gp, gc = torch.autograd.grad(img, (pts, col), torch.tensor(g, device="cuda"))
        ref, rp, rc, n = pyoracle.diff_run(scene, W, H, points=moved, colors=col.detach().cpu().numpy(), grad_image=g,
                                           samples=rows, double=False)
        assert r.crossings() == n
        np.testing.assert_allclose(img.detach().cpu().numpy(), ref, rtol=0, atol=1e-4)
        for a, b in ((gp, rp), (gc, rc)):
            a = a.cpu().numpy().astype(np.float64)
            assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b) + 1e-6
    finally:
        r.close()


def test_nothing_is_filled_after_the_last_crossing():
    """A lone segment from top to bottom opens its winding and never closes it."""
    vg = scanline.VGContainer()
    vg.addPath(0, scanline.rgba(0, 0, 0, 255))
    vg.addLinear((20.5, -1.0), (20.5, 9.0))
    r = diff.DiffRenderer(vg, 64, 8, samples=4)
    try:
        img = r.forward_raw(r.points0, r.colors0, keep=False)
        assert torch.equal(img, torch.ones_like(img))
    finally:
        r.close()
