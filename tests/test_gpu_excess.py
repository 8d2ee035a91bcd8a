"""Excess-plane sweeps (sgm_excess.h) against the one-aggregate schedule, bit for
bit: every wave shape (16, 32 and 64 lanes per line, 4 to 20 disparities per
lane) at full and partly padded rows, uint8 and uint16 costs, one plane per path
and per pair of opposite paths, 4 and 8 paths, penalties up to the byte bound,
lines shorter than a prefetch window and images one line wide in a wave group."""
import numpy as np
import pytest

from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu

# planes of opposite pairs start at this many cells of both matching directions
# (volumes beyond 1 GiB with nine bytes per cell)
PAIR_CELLS = (1 << 30) // 9

CENSUS, AD, GRADIENT, ZNCC, ZNCC32 = range(5)

CASES = [
    # (w, h, D, minD, window, cost, dirs, p1, p2, edge, masks)
    # every wave shape of the single sweeps: padded rows of 64 .. 1024 cells
    (90, 41, 3, 0, (5, 5), CENSUS, 8, 4, 24, 32, False),
    (131, 70, 64, -9, (9, 7), CENSUS, 8, 10, 120, 32, True),
    (140, 53, 65, 4, (9, 7), CENSUS, 8, 10, 127, 32, True),
    (261, 50, 192, 0, (9, 7), CENSUS, 8, 10, 128, 32, False),
    (300, 47, 193, -30, (7, 7), AD, 8, 8, 48, 32, True),
    (350, 40, 256, 0, (9, 7), CENSUS, 8, 10, 193, 0, False),
    (420, 33, 257, 7, (11, 11), GRADIENT, 8, 20, 120, 255, False),
    (430, 31, 320, 0, (9, 7), CENSUS, 8, 0, 1, 32, False),
    (440, 35, 321, -6, (9, 7), CENSUS, 8, 10, 120, 32, True),
    (460, 30, 385, 0, (5, 5), ZNCC, 8, 4, 96, 32, False),
    (540, 30, 512, 0, (9, 7), CENSUS, 8, 10, 120, 32, False),
    (600, 24, 513, -11, (5, 5), CENSUS, 8, 4, 24, 32, True),
    (640, 24, 577, 0, (9, 7), CENSUS, 8, 10, 120, 32, False),
    (700, 24, 641, 5, (7, 7), AD, 8, 8, 48, 32, False),
    (720, 22, 700, 31, (5, 5), CENSUS, 8, 4, 24, 32, False),
    (800, 22, 768, 0, (9, 7), CENSUS, 8, 10, 120, 32, False),
    (1050, 22, 1024, 0, (9, 7), CENSUS, 8, 10, 120, 32, False),
    # uint16 costs, the largest penalty (P1 above P2: P2 becomes P1 + 1)
    (150, 60, 48, -3, (7, 7), ZNCC32, 8, 12, 150, 32, True),
    (280, 45, 192, 0, (7, 7), ZNCC32, 8, 254, 3, 32, False),
    (340, 40, 300, 2, (5, 5), ZNCC32, 8, 12, 150, 32, False),
    (90, 40, 60, 0, (3, 3), CENSUS, 8, 246, 3, 32, False),
    # 4 paths: planes in the room of two partial aggregates
    (201, 81, 97, -13, (11, 11), AD, 4, 20, 120, 32, True),
    (160, 60, 200, 0, (9, 7), CENSUS, 4, 10, 255, 32, False),
    (150, 60, 80, 0, (7, 7), ZNCC32, 4, 12, 150, 32, False),
    # short and narrow: fewer steps than a window, fewer lines than a wave's
    (15, 9, 8, 0, (3, 3), CENSUS, 8, 4, 24, 32, False),
    (300, 9, 64, 0, (5, 5), CENSUS, 8, 4, 24, 32, False),
    (13, 260, 16, -4, (5, 5), CENSUS, 8, 4, 24, 32, True),
    # planes of opposite pairs, by shape
    (1003, 931, 64, 0, (9, 7), CENSUS, 8, 10, 120, 32, True),
    (701, 670, 128, -5, (9, 7), CENSUS, 8, 10, 127, 32, False),
    (650, 479, 192, 0, (5, 5), CENSUS, 8, 4, 63, 32, False),
    (641, 366, 250, 3, (9, 7), CENSUS, 8, 10, 120, 32, True),
    (623, 303, 320, 0, (9, 7), CENSUS, 8, 10, 120, 32, False),
    (610, 257, 350, -17, (9, 7), CENSUS, 8, 10, 64, 32, False),
    (640, 210, 512, 0, (9, 7), CENSUS, 8, 10, 120, 0, False),
    (901, 117, 580, 0, (5, 5), CENSUS, 8, 4, 24, 32, False),
    (1000, 94, 640, 0, (9, 7), CENSUS, 8, 10, 120, 32, False),
    (1100, 79, 700, 0, (9, 7), CENSUS, 8, 10, 120, 32, True),
    (1200, 50, 1024, 0, (5, 5), CENSUS, 8, 4, 24, 32, False),
    (610, 520, 190, 0, (7, 7), ZNCC32, 8, 8, 48, 32, False),
    (610, 310, 320, 0, (7, 7), ZNCC32, 8, 8, 120, 32, False),
    (60, 4700, 250, 0, (9, 7), AD, 8, 10, 120, 32, False),
]


@pytest.mark.parametrize("cfg", CASES, ids=[str(i) for i in range(len(CASES))])
def test_excess_planes_equal_the_aggregate(cfg):
    w, h, D, md, (ww, wh), cost, dirs, p1, p2, edge, masks = cfg
    p = sgm.SgmParams(window_w=ww, window_h=wh, disparities=D, min_disparity=md, cost=cost, p1=p1,
                      p2=p2, edge_scale=edge, directions=dirs, aggregate_bytes=0,
                      census_weight=500, ad_truncation=30, gradient_truncation=60, reserved=0,
                      uniqueness=0.03, lr_threshold=1.0)
    left, right, _ = synth.stereo_pair(w, h, min(D, w - 2), md, seed=D + w)
    vl = vr = None
    if masks:
        rng = np.random.default_rng(w)
        vl = (rng.random((h, w)) > 0.05).astype(np.uint8)
        vr = (rng.random((h, w)) > 0.05).astype(np.uint8)
    out = {}
    for name in ("sequential", "auto"):
        ctx = sgm.Context(0)
        try:
            ctx.sweeps(name)
            print("excess", name, cfg, flush=True)
            plan = ctx.plan(p, w, h)
            assert plan["sweeps"] == (1 if name == "sequential" else 3 if dirs == 8 else 2)
            ctx.set_profiling(True)
            out[name] = ctx.match_pair(p, left, right, vl, vr)
            ran = ctx.profile()["device_kernel_milliseconds"]
            assert ("path_excess" in ran) == (name == "auto"), ran
        finally:
            ctx.close()
    a, b = out["auto"], out["sequential"]
    for k in ("checked", "dl", "dr"):
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k
    for k in ("reasons", "boundary"):
        assert np.array_equal(a[k], b[k]), k
    assert a["stats"] == b["stats"]


def test_pair_cases_reach_the_pair_sweeps():
    for (w, h, D, _, _, _, dirs, p1, p2, _, _) in CASES[27:]:
        Dp = -(-D // 64) * 64
        assert dirs == 8 and 2 * max(p1 + 1, p2) <= 255 and 2 * w * h * Dp > PAIR_CELLS
    for (w, h, D, *_rest) in CASES[:27]:
        assert 2 * w * h * (-(-D // 64) * 64) <= PAIR_CELLS
