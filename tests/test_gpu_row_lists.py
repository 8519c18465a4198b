"""GPU: the compositors' row lists and the scans, against the oracle, image bytes equal.

Path and row counts around the groups of 64 that a wave walks, path counts around the size
where one block stops scanning alone (16384), paths above, below and across the canvas,
paths without visible curves, and batches whose scenes start inside a group of rows, one of
them with far more paths than the others.
"""
import numpy as np
import pytest

import pyoracle
import scanline
from scanline import VGContainer, rgba

pytestmark = pytest.mark.gpu


def scene(W, H, P, seed):
    rng = np.random.default_rng(seed)
    vg = VGContainer(W, H)
    for k in range(P):
        kind = rng.integers(0, 10)
        y = rng.uniform(-6, H + 6)
        h = H * 1.5 if kind == 0 else rng.uniform(0.2, 9)
        if kind == 1:
            y = -300.0 if k & 1 else H + 300.0  # nothing on the canvas
        x, w = rng.uniform(-8, W), rng.uniform(0.5, W / 2 + 2)
        vg.addPath(k & 1, rgba(*rng.integers(0, 256, 3), int(rng.integers(20, 256))))
        vg.addPolygon([(x, y), (x + w, y + 0.3 * h), (x + 0.4 * w, y + h)])
    return vg.arrays()


def oracle(a, W, H, spp=16):
    return pyoracle.run(a, W, H, spp, srgb=True, ms=False, keep=False)


def check(r, a, W, H):
    print("row lists:", W, H, a.n_paths, flush=True)
    ref = oracle(a, W, H)
    r.setSamples(16)
    r.enableSRGBCorrection(True)
    r.setMultisampleOutput(False)
    r.resizeOutputBuffer(W, H)
    r.setInputTransform(np.eye(4, dtype=np.float32))
    r.addVg(a)
    for rep in range(2):  # the frame that reads its sizes, then one that does not
        r.rasterize()
        assert r.elementNumber() == ref.counts()
        np.testing.assert_array_equal(r.output(), ref.get("image").reshape(H, W, 4))


@pytest.mark.parametrize("P", [1, 2, 63, 64, 65, 128, 129, 700])
@pytest.mark.parametrize("H", [1, 2, 3, 126, 127, 128, 129, 131, 300])
def test_paths_and_rows_around_64(rasterizer, P, H):
    rasterizer.dumpDebugData(False)
    check(rasterizer, scene(40, H, P, 7 * P + H), 40, H)


@pytest.mark.parametrize("P", [16383, 16384, 16385])
def test_scans_around_one_block(rasterizer, P):
    rasterizer.dumpDebugData(False)
    check(rasterizer, scene(150, 200, P, P), 150, 200)


def test_row_order_dump(rasterizer):
    a = scene(90, 200, 150, 5)
    rasterizer.dumpDebugData(True)
    try:
        check(rasterizer, a, 90, 200)
        info, cnt = rasterizer.dump("bucket_info"), rasterizer.dump("bucket_items")
        keys, order = rasterizer.dump("row_keys"), rasterizer.dump("row_list")
        beg, end = rasterizer.dump("row_beg"), rasterizer.dump("row_end")
        full = np.flatnonzero(cnt.ravel())
        want = full[np.lexsort((info[full, 0], info[full, 1]))]
        np.testing.assert_array_equal(order.ravel(), want)
        np.testing.assert_array_equal(keys.ravel(), info[want, 1])
        for r in range(100):
            rows = np.flatnonzero(info[want, 1] == r)
            assert (end.ravel()[r] - beg.ravel()[r] == len(rows)) and (not len(rows) or beg.ravel()[r] == rows[0])
    finally:
        rasterizer.dumpDebugData(False)


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_batches_of_uneven_scenes(seed):
    rng = np.random.default_rng(seed)
    sizes = [(int(rng.integers(1, 90)), int(rng.integers(1, 150))) for _ in range(70)]
    paths = [int(rng.integers(1, 12)) for _ in sizes]
    paths[33 + seed] = 900  # one scene holds most of the paths
    sizes[10] = (30, 700)   # and one spans many groups of rows
    scenes = [scene(w, h, p, 100 * seed + i) for i, ((w, h), p) in enumerate(zip(sizes, paths))]
    print("batch", seed, sum(paths), flush=True)
    b = scanline.BatchRasterizer(scenes, sizes, [16] * len(scenes))
    try:
        for rep in range(2):
            b.render()
            for i, (w, h) in enumerate(sizes):
                np.testing.assert_array_equal(b.output(i), oracle(scenes[i], w, h).get("image").reshape(h, w, 4))
    finally:
        b.close()
