"""Disparity outputs of the device entry point when a call is interrupted: the
caller's maps keep what they held (they are written by a call that ends well)."""
import threading
import time

import numpy as np
import pytest

from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu

INTERRUPTED = -9


@pytest.mark.parametrize("plan", ["resident", "esgm", "streamed"])
def test_interrupted_call_leaves_the_disparity_maps(plan):
    w, h, D = 1600, 400, 128
    left, right, _ = synth.stereo_pair(w, h, D, 0, seed=71)
    p = sgm.SgmParams(window_w=9, window_h=7, disparities=D, min_disparity=0, cost=0, p1=8, p2=96,
                      edge_scale=32, directions=8, aggregate_bytes=0, census_weight=500,
                      ad_truncation=30, gradient_truncation=60, reserved=0, uniqueness=0.03,
                      lr_threshold=1.0)
    ctx = sgm.Context(0)
    try:
        # streamed: one-row strips recomputed strip by strip, hundreds of passes that
        # each end in the selection of their row
        ctx.plan_mode(plan, 1 if plan == "streamed" else 64)
        if plan == "streamed":
            ctx.aggregate_storage("recompute", None, 2 * w * D * 2)
            assert ctx.plan(p, w, h)["block_rows"] == 1
        dleft, dright = ctx.alloc(w * h).upload(left), ctx.alloc(w * h).upload(right)
        held = np.full(w * h, -7.5, np.float32)
        maps = [ctx.alloc(4 * w * h).upload(held) for _ in range(3)]
        if plan != "streamed":
            ctx.interrupt()  # before the call: it stops at its first check
        later = threading.Thread(target=lambda: (time.sleep(0.5), ctx.interrupt()))
        if plan == "streamed":
            later.start()
        print("interrupted outputs", plan, flush=True)
        with pytest.raises(sgm.SgmError) as e:
            ctx.match_pair_device(p, dleft.ptr, dright.ptr, w, h, maps[0].ptr, d_dl=maps[1].ptr,
                                  d_dr=maps[2].ptr)
        assert e.value.code == INTERRUPTED
        if plan == "streamed":
            later.join()
        ctx.synchronize()
        for m in maps:
            assert np.array_equal(m.download(np.float32, w * h), held)
        for b in [dleft, dright] + maps:
            b.free()
    finally:
        ctx.close()
