"""Band cost kernel (sgm_cost.h): census, AD-census and census-gradient cost
volumes against the oracle's, cell for cell, over every wave shape, one- and
two-word descriptors, uint8 and uint16 volumes, both matching directions,
segment remainders, weights and truncations up to the numerator bound."""
import numpy as np
import pytest

from oracle import oracle as O
from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu

CASES = [
    # (w, h, D, minD, window, cost, aggregate_bytes, weight, ad cap, gradient cap, masks)
    (47, 15, 3, 0, (3, 3), 1, 0, 500, 30, 60, False),
    (131, 24, 64, -9, (11, 11), 0, 0, 500, 30, 60, True),
    (129, 17, 70, 4, (9, 7), 2, 0, 500, 30, 60, True),
    (257, 16, 150, -20, (11, 9), 1, 0, 0, 1, 60, False),
    (260, 16, 200, 0, (9, 7), 2, 0, 1000, 30, 1020, False),
    (300, 14, 300, -33, (11, 11), 1, 0, 300, 255, 60, True),
    (330, 14, 350, 7, (9, 7), 2, 0, 700, 30, 17, False),
    (450, 14, 450, 0, (5, 5), 1, 0, 500, 4000, 60, False),
    (470, 14, 512, -40, (11, 11), 2, 0, 500, 30, 60, False),
    (540, 13, 530, 0, (9, 7), 0, 0, 500, 30, 60, True),
    (600, 13, 600, 12, (7, 7), 1, 0, 500, 30, 60, False),
    (640, 13, 640, 0, (5, 5), 0, 0, 500, 30, 60, False),
    (660, 13, 700, 31, (11, 11), 0, 0, 500, 30, 60, False),
    (700, 13, 1000, -60, (7, 7), 2, 0, 500, 30, 60, False),
    # uint16 volumes (32-bit sums)
    (150, 20, 65, 0, (9, 7), 0, 4, 500, 30, 60, True),
    (280, 15, 257, -5, (11, 11), 1, 4, 500, 30, 60, False),
    (700, 13, 640, 3, (9, 7), 2, 4, 500, 30, 60, False),
    # numerators just below 2^31
    (120, 15, 50, 0, (11, 11), 1, 0, 1000, 17800, 60, False),
]


@pytest.mark.parametrize("cfg", CASES, ids=[str(i) for i in range(len(CASES))])
def test_cost_volume_equals_the_oracle(cfg):
    w, h, D, md, (ww, wh), cost, agg, weight, ad, grad, masks = cfg
    left, right, _ = synth.stereo_pair(w, h, min(D, w - 2), md, seed=D)
    valid = None
    if masks:
        valid = (np.random.default_rng(w).random((h, w)) > 0.1).astype(np.uint8)
    op = O.params(window_w=ww, window_h=wh, disparities=D, min_disparity=md, cost=cost, p1=10,
                  p2=120, aggregate_bytes=agg, census_weight=weight, ad_truncation=ad,
                  gradient_truncation=grad, lr_threshold=1.0)
    p = sgm.SgmParams(**{f: getattr(op, f) for f, _ in sgm.SgmParams._fields_})
    images = (left.reshape(-1), right.reshape(-1))
    census = [O.census(g, w, h, ww, wh) for g in images]
    texture = [O.texture(g, w, h, ww, wh, valid) for g in images]
    print("cost case", cfg, flush=True)
    ctx = sgm.Context(0)
    try:
        ctx.keep_volumes(True)
        ctx.match_pair(p, left, right, valid, valid)
        for d in (0, 1):
            a, b = d, 1 - d
            want = O.match(op, census[a], census[b], images[a], images[b], texture[a], texture[b],
                           w, h, d, volumes=True)
            got, _ = ctx.read_volumes(d, w * h, D)
            assert np.array_equal(got, want[4]), "direction %d" % d
    finally:
        ctx.close()
