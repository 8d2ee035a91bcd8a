"""Images wider than 2^25 / D columns take the kernels that narrower ones take (band
costs, excess planes), with the results of the one-aggregate schedule."""
import numpy as np
import pytest

from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu


# (width, height, disparities, P2): lines of a wave 1, 2 and 4 rows apart
@pytest.mark.parametrize("w,h,D,p2", [(70000, 10, 500, 24), (70000, 9, 500, 150), (110000, 11, 300, 24),
                                      (135000, 10, 250, 150), (36000, 8, 1000, 24)])
def test_wide_images_equal_the_aggregate(w, h, D, p2):
    p = sgm.SgmParams(window_w=5, window_h=5, disparities=D, min_disparity=-3, cost=0, p1=10, p2=p2,
                      edge_scale=32, directions=8, aggregate_bytes=0, census_weight=500,
                      ad_truncation=30, gradient_truncation=60, reserved=0, uniqueness=0.03,
                      lr_threshold=1.0)
    left, right, _ = synth.stereo_pair(w, h, D, -3, seed=D)
    out = {}
    for schedule in ("sequential", "auto"):
        ctx = sgm.Context(0)
        try:
            ctx.sweeps(schedule)
            ctx.set_profiling(True)
            print("wide", w, h, D, p2, schedule, flush=True)
            out[schedule] = ctx.match_pair(p, left, right)
            ran = ctx.profile()["device_kernel_milliseconds"]
            if schedule == "auto":
                assert "path_excess" in ran and "path_cost" in ran and "cost" not in ran, ran
        finally:
            ctx.close()
    a, b = out["auto"], out["sequential"]
    for k in ("checked", "dl", "dr"):
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k
    for k in ("reasons", "boundary"):
        assert np.array_equal(a[k], b[k]), k
    assert a["stats"] == b["stats"]
