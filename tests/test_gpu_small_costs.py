"""Cost volumes of small images without planes: a thread per four cells below a number
of waves, row segments from there on; the results are those of the row segments (which
kept volumes always take)."""
import numpy as np
import pytest

from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu


# (w, h, D, window, cost, bytes of a sum, row segments)
@pytest.mark.parametrize("w,h,D,window,cost,sums,segments", [
    (61, 25, 640, (9, 9), 1, 4, False), (185, 14, 700, (7, 7), 2, 2, False),
    (100, 40, 320, (11, 11), 1, 4, False), (120, 70, 60, (9, 7), 0, 4, False),
    (150, 115, 64, (11, 11), 0, 2, False), (150, 118, 64, (11, 11), 0, 2, True),
    (130, 64, 1000, (5, 5), 1, 4, True), (140, 84, 500, (9, 7), 2, 2, True)])
def test_small_images_take_the_shorter_kernel(w, h, D, window, cost, sums, segments):
    p = sgm.SgmParams(window_w=window[0], window_h=window[1], disparities=D, min_disparity=-4,
                      cost=cost, p1=10, p2=400, edge_scale=32, directions=4, aggregate_bytes=sums,
                      census_weight=500, ad_truncation=30, gradient_truncation=60, reserved=0,
                      uniqueness=0.03, lr_threshold=1.0)
    left, right, _ = synth.stereo_pair(w, h, max(8, min(D, w - 2)), -4, seed=D)
    out = {}
    for keep in (True, False):
        ctx = sgm.Context(0)
        try:
            ctx.keep_volumes(keep)
            ctx.set_profiling(True)
            print("small costs", w, h, D, window, cost, sums, keep, flush=True)
            out[keep] = ctx.match_pair(p, left, right)
            ran = ctx.profile()["device_kernel_milliseconds"]
            assert ("path_cost" in ran) == (keep or segments) and ("cost" in ran) != ("path_cost" in ran)
        finally:
            ctx.close()
    for k in ("checked", "dl", "dr"):
        assert np.array_equal(out[True][k].view(np.uint32), out[False][k].view(np.uint32)), k
    assert out[True]["stats"] == out[False]["stats"]
