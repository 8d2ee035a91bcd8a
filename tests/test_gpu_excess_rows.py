"""Excess-plane sweeps whose rows fill their padded length exactly (and a few that do
not), in every wave shape: the ranges whose rows leave lanes of a line idle (448, 576, 704, 832, 896 and
960 disparities) have a real cell beside the idle lanes.  Single planes, pairs
of opposite paths and 32-bit sums, in the caches and (volumes beyond 1 GiB) with
the accesses that pass them; each equals the one-aggregate schedule bit for bit."""
import numpy as np
import pytest

from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu

GIB = 1 << 30
SPARE = [448, 576, 704, 832, 896, 960]  # padded rows that leave lanes idle
SHAPES = [64, 128, 192, 256, 320, 384, 512, 640, 768, 1024]  # one row per further shape


def size_of(D, cells, wide):
    """A width past the range and a height that takes `cells` cells, both directions;
    up to 512 disparities at least half the width (longer images go by another rule)."""
    w = (max(D + 90, 620) if cells else D + 60) | 1
    return w, max(w // 2 + 1 if D <= 512 and not wide else 24, cells // (2 * w * D) + 1)


# (name, D, cells of both directions, P2, bytes of a sum, planes, streamed)
CASES = ([("pairs", D, GIB // 9, 120, 2, 4, False) for D in SPARE + [300, 350, 500]] +
         [("pairs streamed", D, GIB // 5, 120, 2, 4, True) for D in SPARE + SHAPES] +
         [("single", D, 0, 150, 2, 8, False) for D in SPARE] +
         [("single streamed", D, GIB // 9, 150, 2, 8, True) for D in SPARE + SHAPES] +
         [("wide", D, 0, 120, 4, 4, False) for D in SPARE] +
         [("wide streamed", D, GIB // 6, 120, 4, 4, True) for D in SPARE + SHAPES])


@pytest.mark.parametrize("case", CASES, ids=["%s-%d" % (c[0].replace(" ", "-"), c[1]) for c in CASES])
def test_full_rows_equal_the_aggregate(case):
    name, D, cells, p2, sums, planes, streamed = case
    w, h = size_of(D, cells, name.startswith("wide"))
    p = sgm.SgmParams(window_w=9, window_h=7, disparities=D, min_disparity=0, cost=0, p1=10, p2=p2,
                      edge_scale=32, directions=8, aggregate_bytes=sums, census_weight=500,
                      ad_truncation=30, gradient_truncation=60, reserved=0, uniqueness=0.03,
                      lr_threshold=1.0)
    cost = 1 if sums == 2 else 2
    # the rules on sizes that choose the planes and the cache policy
    padded = -(-D // 64) * 64
    assert (2 * w * h * padded * 9 > GIB and 2 * p2 <= 255) == name.startswith("pairs") or sums == 4
    assert (2 * w * h * padded * (cost + planes) > GIB) == streamed
    # most pixels near the top of the range, beside the idle lanes
    left, right, _ = synth.stereo_pair(w, h, D, 0, seed=D)
    shift = D - 2
    right = np.array(right)
    right[:, : w - shift] = np.array(left)[:, shift:]
    out = {}
    for schedule in ("sequential", "auto"):
        ctx = sgm.Context(0)
        try:
            ctx.sweeps(schedule)
            print("full rows", name, D, w, h, schedule, flush=True)
            ctx.set_profiling(True)
            out[schedule] = ctx.match_pair(p, left, right)
            ran = ctx.profile()["device_kernel_milliseconds"]
            assert ("path_excess" in ran) == (schedule == "auto"), ran
        finally:
            ctx.close()
    a, b = out["auto"], out["sequential"]
    for k in ("checked", "dl", "dr"):
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k
    for k in ("reasons", "boundary"):
        assert np.array_equal(a[k], b[k]), k
    assert a["stats"] == b["stats"]


def test_rows_of_20_bytes_a_lane_cost_what_other_rows_do():
    """One plane per path beyond the caches: a cell of the 320-disparity shape (20
    bytes a lane, two accesses) takes no longer than 1.3 of a 384-disparity one."""
    per_cell = {}
    for D in (320, 384):
        w, h = 1600, 900
        p = sgm.SgmParams(window_w=9, window_h=7, disparities=D, min_disparity=0, cost=0, p1=10,
                          p2=150, edge_scale=32, directions=8, aggregate_bytes=0,
                          census_weight=500, ad_truncation=30, gradient_truncation=60, reserved=0,
                          uniqueness=0.03, lr_threshold=1.0)
        left, right, _ = synth.stereo_pair(w, h, D, 0, seed=D)
        ctx = sgm.Context(0)
        try:
            ctx.match_pair(p, left, right)
            ctx.set_profiling(True)
            runs = []
            for _ in range(5):
                ctx.profile()
                ctx.match_pair(p, left, right)
                runs.append(ctx.profile()["device_kernel_milliseconds"]["path_excess"]["total_ms"])
            per_cell[D] = min(runs) / D
        finally:
            ctx.close()
    print("excess sweeps, us per disparity:", per_cell, flush=True)
    assert per_cell[320] <= 1.3 * per_cell[384], per_cell
