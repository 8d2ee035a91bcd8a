"""Whole-image line sweeps of the compact plan: their results equal the resident
plan's bit for bit for every line shape (lanes per line, disparities per lane),
with ragged last waves, images narrower than a wave of lines, signed ranges,
masked and textureless input, proposal counts up to the most that fit, and P2 on
both sides of what 16-bit sums hold."""
import numpy as np
import pytest

from pose_amd import sgm, synth
from tests.test_gpu_esgm import esgm
from tests.test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu


def _params(D, md, directions, **over):
    f = dict(window_w=9, window_h=7, disparities=D, min_disparity=md, cost=0, p1=8, p2=96,
             edge_scale=32, directions=directions, aggregate_bytes=0, census_weight=500,
             ad_truncation=30, gradient_truncation=60, reserved=0, uniqueness=0.03,
             lr_threshold=1.0)
    f.update(over)
    return sgm.SgmParams(**f)


# (w, h, D, min disparity, directions, pool, changed parameters)
CASES = [
    (37, 19, 3, 0, 8, 4, {}),
    (5, 41, 4, -1, 4, 1, {"window_w": 3, "window_h": 3}),
    (70, 23, 63, 0, 8, 4, {}),
    (130, 33, 64, -7, 8, 2, {"window_w": 5, "window_h": 5}),
    (133, 30, 65, 3, 8, 3, {"edge_scale": 0}),
    (141, 35, 128, 0, 4, 4, {"p1": 0, "p2": 1}),
    (150, 29, 160, -20, 8, 2, {"window_w": 3, "window_h": 11}),
    (171, 26, 192, 0, 8, 1, {}),
    (200, 22, 250, 0, 8, 4, {"p1": 100, "p2": 255}),
    (190, 21, 257, -9, 4, 2, {}),
    (210, 18, 320, 0, 8, 2, {}),
    (240, 17, 340, 5, 8, 3, {}),
    (230, 16, 384, 0, 4, 2, {}),
    (260, 15, 448, -30, 8, 2, {}),
    (280, 14, 511, 0, 8, 1, {}),
    (120, 31, 90, 0, 8, 2, {"p1": 600, "p2": 7600}),
    (110, 33, 80, 0, 4, 2, {"p1": 900, "p2": 9216}),
    (110, 33, 80, 0, 4, 2, {"p1": 900, "p2": 12000}),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_lines_equal_resident(gpu_context, case):
    w, h, D, md, directions, pool, over = CASES[case]
    p = _params(D, md, directions, **over)
    left, right, _ = synth.stereo_pair(w, h, max(D, 8), md, seed=900 + case)
    # a constant patch: ties everywhere, so both certified and verified pixels
    left, right = np.array(left), np.array(right)
    left[: h // 2, : w // 3] = 90
    right[: h // 2, : w // 3] = 90
    rng = np.random.default_rng(case)
    vl = rng.random((h, w)) > 0.05 if case % 3 == 0 else None
    vr = rng.random((h, w)) > 0.05 if case % 3 == 0 else None
    if vl is not None:
        vl, vr = vl.astype(np.uint8), vr.astype(np.uint8)
    want = gpu_context.match_pair(p, left, right, vl, vr)
    got, counts = esgm(gpu_context, p, left, right, vl, vr, rows=h, pool=pool,
                       what="lines case %d D %d" % (case, D))
    assert_same(got, want, "case %d" % case)
    for side in ("left", "right"):
        assert sum(counts[side]) == w * h
