"""Census kernel (sgm_census.hip): every window, image widths of every remainder
of four, several tiles and remainders of one, masks, against the oracle: census
cost volumes cell for cell (the descriptors and the texture mask decide them)
and the results of ZNCC matching (the window sums decide them)."""
import numpy as np
import pytest

from oracle import oracle as O
from pose_amd import sgm, synth
from tests.test_gpu_parity import assert_same, to_sgm

pytestmark = pytest.mark.gpu

SIDES = (3, 5, 7, 9, 11)


@pytest.mark.parametrize("wh", SIDES)
@pytest.mark.parametrize("ww", SIDES)
def test_census_windows(gpu_context, ww, wh):
    w, h, D = 60 + ww + wh // 2, 14 + 2 * wh, 5
    left, right, _ = synth.stereo_pair(w, h, D, 0, seed=ww * 16 + wh)
    left, right = np.array(left), np.array(right)
    left[3:12, 5:30] = 77  # no texture
    valid = (np.random.default_rng(ww).random((h, w)) > 0.1).astype(np.uint8)
    op = O.params(window_w=ww, window_h=wh, disparities=D, min_disparity=-1, cost=0, p1=10,
                  p2=120, lr_threshold=1.0)
    images = (left.reshape(-1), right.reshape(-1))
    census = [O.census(g, w, h, ww, wh) for g in images]
    texture = [O.texture(g, w, h, ww, wh, valid) for g in images]
    print("census window", ww, wh, w, h, flush=True)
    ctx = sgm.Context(0)
    try:
        ctx.keep_volumes(True)
        ctx.match_pair(to_sgm(op), left, right, valid, valid)
        for d in (0, 1):
            a, b = d, 1 - d
            want = O.match(op, census[a], census[b], images[a], images[b], texture[a], texture[b],
                           w, h, d, volumes=True)
            got, _ = ctx.read_volumes(d, w * h, D)
            assert np.array_equal(got, want[4]), "direction %d" % d
    finally:
        ctx.close()
    op = O.params(window_w=ww, window_h=wh, disparities=D, min_disparity=-1, cost=3, p1=10,
                  p2=120, lr_threshold=1.0)
    want = O.compute(op, left, right, w, h, valid, valid)
    assert_same(gpu_context.match_pair(to_sgm(op), left, right, valid, valid), want,
                "zncc window %dx%d" % (ww, wh))
