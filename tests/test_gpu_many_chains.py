"""GPU: frames whose cubic chains are too many to take several lanes each.

How many length bins get several lanes is decided by the cuts in them: all of the rule's,
the first ones, or none.  Scenes of curves of chosen lengths reach each outcome under each
rule by the frame's cuts; every intersection is compared with the oracle, bit for bit, and the
image.  The stage's time is compared between a few and many long chains: lanes of their own
take a GPU's time in proportion, a lane each hardly more.
"""
import numpy as np
import pytest

import pyoracle
import scanline
from scanline.scene import SceneArrays, rgba

pytestmark = pytest.mark.gpu


def curves(W, groups, seed):
    """groups: (count, length): cubics of that extent each way, closed by a line."""
    rng = np.random.default_rng(seed)
    v = []
    for n, L in groups:
        o = rng.uniform(0, W - L, (n, 1, 2))
        bend = np.array([[0, 0], [0.3, 0.5], [0.8, 0.6], [1, 1], [1, 1], [0, 0]]) + np.zeros((n, 1, 1))
        bend[:, 1:3] += rng.uniform(-0.1, 0.1, (n, 2, 2))
        v.append((o + L * bend).reshape(-1, 2))
    n = sum(g[0] for g in groups)
    pos = np.stack([6 * np.arange(n), 6 * np.arange(n) + 4], 1).reshape(-1)
    return SceneArrays(np.concatenate(v), pos, [4, 2] * n, np.repeat(np.arange(n), 2), [-1.0] * (2 * n),
                       np.arange(n) & 1, [rgba(40, 90, 160, 60)] * n)


def setup(r, W):
    r.setSamples(8)
    r.enableSRGBCorrection(True)
    r.setMultisampleOutput(False)
    r.resizeOutputBuffer(W, W)
    r.setInputTransform(np.eye(4, dtype=np.float32))


@pytest.mark.parametrize("groups,limits", [
    ([(2500, 24)], (0, 1 << 18)),                          # up to 2^18 cuts: all, ...
    ([(9000, 60)], (1 << 18, 1 << 21)),                    # no chains: the pieces are too short
    ([(4000, 120)], (1 << 18, 1 << 21)),                   # none
    ([(40, 400), (4000, 120)], (1 << 18, 1 << 21)),        # all, for the long ones' sake
    ([(4, 180), (5000, 140)], (1 << 18, 1 << 21)),         # the first bins
    ([(3200, 420)], (1 << 21, 5 << 20)),                   # none
    ([(60, 700), (2600, 450)], (1 << 21, 5 << 20)),        # the first bins
    ([(2400, 900)], (1 << 21, 5 << 20)),                   # none
    ([(3600, 900)], (5 << 20, 1 << 24)),                   # none
    ([(500, 980), (4000, 600)], (5 << 20, 1 << 24))])      # the first bins
def test_intersections(rasterizer, groups, limits):
    W = 1000
    a = curves(W, groups, len(groups) + groups[0][0])
    print("many chains:", groups, a.n_curves, flush=True)
    r = rasterizer
    setup(r, W)
    r.dumpDebugData(True)
    try:
        r.addVg(a)
        r.rasterize()
        ref = pyoracle.run(a, W, W, 8, srgb=True, ms=False)
        F = r.elementNumber()["curve_fragment"]
        assert limits[0] < F <= limits[1], F
        np.testing.assert_array_equal(r.dump("ts"), ref.get("ts"))
        np.testing.assert_array_equal(r.output(), ref.get("image").reshape(W, W, 4))
    finally:
        r.dumpDebugData(False)


def test_time_of_many_long_chains(rasterizer):
    r, W = rasterizer, 512
    setup(r, W)
    r.dumpDebugData(False)
    ms = {}
    r.enableStepTiming(True)
    try:
        for n in (2250, 18000):
            r.addVg(curves(W, [(n, 400)], n))
            t = []
            for _ in range(6):
                r.rasterize()
                t.append(r.stepTiming()["intersect"])
            ms[n] = min(t)
    finally:
        r.enableStepTiming(False)
    print("many chains:", ms, flush=True)
    assert ms[18000] <= 2.5 * ms[2250]
