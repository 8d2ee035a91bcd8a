"""One session over changing options: path counts, penalties, sum widths and sizes
follow each other on one context (whose buffers and wave orders stay), and every
result equals that of a fresh context under the one-aggregate schedule."""
import numpy as np
import pytest

from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu


def params(D, dirs, p2, sums, cost=0):
    return sgm.SgmParams(window_w=9, window_h=7, disparities=D, min_disparity=0, cost=cost, p1=10,
                         p2=p2, edge_scale=32, directions=dirs, aggregate_bytes=sums,
                         census_weight=500, ad_truncation=30, gradient_truncation=60, reserved=0,
                         uniqueness=0.03, lr_threshold=1.0)


# (w, h, [(D, paths, P2, bytes of a sum, cost)]): at one size four paths, the four
# pairs of eight, and eight single paths; 1003x931 D=64 has its 16-bit planes in pairs
SESSIONS = [
    (211, 130, [(64, 4, 120, 4, 0), (64, 8, 120, 4, 0), (64, 4, 120, 4, 0), (64, 8, 120, 2, 0),
                (64, 4, 200, 2, 0), (64, 8, 180, 2, 0), (64, 8, 180, 4, 0), (64, 8, 60, 4, 0)]),
    (160, 97, [(100, 8, 120, 4, 0), (100, 4, 120, 4, 4), (300, 8, 120, 4, 0), (300, 4, 90, 4, 0),
               (300, 8, 120, 2, 4), (100, 4, 255, 2, 4), (100, 8, 100, 4, 4)]),
    (1003, 931, [(64, 4, 120, 2, 0), (64, 8, 120, 2, 0), (64, 4, 120, 2, 0), (64, 8, 128, 2, 0),
                 (64, 8, 127, 2, 0)]),
]


@pytest.mark.parametrize("session", range(len(SESSIONS)))
def test_results_do_not_depend_on_the_calls_before(session):
    w, h, calls = SESSIONS[session]
    left, right, _ = synth.stereo_pair(w, h, 60, 0, seed=40 + session)
    one = sgm.Context(0)
    try:
        for i, (D, dirs, p2, sums, cost) in enumerate(calls):
            p = params(D, dirs, p2, sums, cost)
            print("session", session, "call", i, calls[i], flush=True)
            got = one.match_pair(p, left, right)
            fresh = sgm.Context(0)
            try:
                fresh.sweeps("sequential")
                want = fresh.match_pair(p, left, right)
            finally:
                fresh.close()
            for k in ("checked", "dl", "dr"):
                assert np.array_equal(got[k].view(np.uint32), want[k].view(np.uint32)), (i, k)
            for k in ("reasons", "boundary"):
                assert np.array_equal(got[k], want[k]), (i, k)
            assert got["stats"] == want["stats"], i
    finally:
        one.close()
