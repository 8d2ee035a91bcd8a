"""Budgets that hold seven bytes of planes per cell and not eight: the planes run in
pairs of opposite paths where two excesses fit a byte, with the results of the
one-aggregate schedule."""
import numpy as np
import pytest

from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu


PLANES, PAIRED = sgm.SWEEPS_PLANES, sgm.SWEEPS_PAIRED


@pytest.mark.parametrize("p2,per_cell,expect", [(120, 7, PLANES), (120, 8, PLANES), (127, 7, PLANES),
                                                (128, 8, PLANES), (120, 6, PAIRED)])
def test_planes_under_a_budget(p2, per_cell, expect):
    w, h, D = 320, 130, 100
    left, right, _ = synth.stereo_pair(w, h, D, 0, seed=78)
    p = sgm.SgmParams(window_w=9, window_h=7, disparities=D, min_disparity=0, cost=0, p1=10, p2=p2,
                      edge_scale=32, directions=8, aggregate_bytes=0, census_weight=500,
                      ad_truncation=30, gradient_truncation=60, reserved=0, uniqueness=0.03,
                      lr_threshold=1.0)
    probe = sgm.Context(0)
    probe.sweeps("sequential")
    plan = probe.plan(p, w, h)
    want = probe.match_pair(p, left, right)
    probe.close()
    cells = 2 * w * h * plan["padded_disparities"]
    base = plan["pair_bytes"] + cells - 2 * cells  # a uint8 cost volume, no aggregates
    ctx = sgm.Context(0, budget_bytes=base + per_cell * cells + (1 << 20))
    try:
        assert ctx.plan(p, w, h)["sweeps"] == expect
        ctx.set_profiling(True)
        got = ctx.match_pair(p, left, right)
        ran = ctx.profile()["device_kernel_milliseconds"]
        assert ("path_excess" in ran) == (expect == sgm.SWEEPS_PLANES), ran
        for k in ("checked", "dl", "dr"):
            assert np.array_equal(got[k].view(np.uint32), want[k].view(np.uint32)), k
        assert got["stats"] == want["stats"]
    finally:
        ctx.close()
