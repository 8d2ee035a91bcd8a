"""Photometric check, subpixel refinement and speckle labelling against the
oracle, bit for bit: every radius with its own instance and the ones beyond, gray
and colour, signed ranges, image widths that leave every byte alignment, speckle
maps over several tiles with few and many links across them."""
import numpy as np
import pytest

from oracle import oracle as O
from pose_amd import sgm, synth
from tests.test_gpu_filters import bits, to_filters
from tests.test_gpu_parity import to_sgm

pytestmark = pytest.mark.gpu


def _same(got, want):
    assert np.array_equal(bits(got["disparity"]), bits(want["disparity"]))
    assert np.array_equal(got["reasons"], want["reasons"])
    for k in O.STAT_FIELDS:
        assert got["stats"][k] == want["stats"][k], k


@pytest.mark.parametrize("window", [3, 5, 7, 9, 11])
@pytest.mark.parametrize("color", [False, True], ids=["gray", "color"])
def test_windows(gpu_context, window, color):
    w, h, D = 131 + window // 2, 70, 24
    left, right, _ = synth.stereo_pair(w, h, D, -3, seed=40 + window)
    op = O.params(window_w=5, window_h=5, disparities=D, min_disparity=-3, lr_threshold=1.0)
    f = O.filters(correlation_window=window, subpixel_refinement=1, speckle_size=15)
    print("photo window", window, color, flush=True)
    if not color:
        want = O.compute_filtered(op, f, left, right, w, h)
        _same(gpu_context.match_pair_filtered(to_sgm(op), to_filters(f), left, right), want)
        return
    rng = np.random.default_rng(window)
    bgr = [np.stack([g, np.roll(g, 1, 0), 255 - g], -1) for g in (left, right)]
    bgr = [np.clip(b.astype(int) + rng.integers(-3, 4, b.shape), 0, 255).astype(np.uint8)
           for b in bgr]
    want = O.compute_filtered(op, f, left, right, w, h, left_bgr=bgr[0], right_bgr=bgr[1])
    _same(gpu_context.match_pair_color(to_sgm(op), left, right, bgr[0], bgr[1], to_filters(f)),
          want)


@pytest.mark.parametrize("conn", [4, 8])
@pytest.mark.parametrize("speckle_range", [0.05, 0.5, 1.0, 40.0])
def test_speckles(gpu_context, conn, speckle_range):
    w, h, D = 203, 101, 20
    left, right, _ = synth.stereo_pair(w, h, D, 0, seed=conn)
    op = O.params(window_w=5, window_h=5, disparities=D, min_disparity=0, lr_threshold=1.0)
    f = O.filters(speckle_connectivity=conn, speckle_range=speckle_range, speckle_size=40,
                  median=1, correlation=-2.0)
    print("speckles", conn, speckle_range, flush=True)
    want = O.compute_filtered(op, f, left, right, w, h)
    _same(gpu_context.match_pair_filtered(to_sgm(op), to_filters(f), left, right), want)
