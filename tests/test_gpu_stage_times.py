"""GPU: stage times.  The rows are ordered in bucket_setup, so the stage that names their
order reads zero, in single frames and under the debug dumps; the others take some time.
"""
import numpy as np
import pytest

import scanline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("debug", [False, True])
@pytest.mark.parametrize("ms", [False, True])
def test_row_order_takes_no_time_of_its_own(rasterizer, ms, debug):
    r = rasterizer
    r.setSamples(8)
    r.setMultisampleOutput(ms)
    r.resizeOutputBuffer(200, 150)
    r.setInputTransform(np.eye(4, dtype=np.float32))
    r.dumpDebugData(debug)
    r.addVg(scanline.generate(scanline.scene.KIND_MIXED, 200, 150, 40, 3))
    r.enableStepTiming(True)
    try:
        r.rasterize()
        t = r.stepTiming()
    finally:
        r.enableStepTiming(False)
        r.dumpDebugData(False)
    print("stage times:", t, flush=True)
    assert t.pop("order_rows") == 0.0
    assert len(t) == 7 and all(0.0 < v < 1000.0 for v in t.values())
