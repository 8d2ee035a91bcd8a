"""Colour-distance census where distances meet their mean exactly or nearly: few levels
(whole distances whose mean is one of them), flat areas (mean 0), the largest distances
and roots that are no whole numbers; bit-exact to the oracle in every window size."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.cases import bgr_gray
from tests.test_gpu_parity import assert_same, to_sgm

pytestmark = pytest.mark.gpu

W, H, D = 110, 48, 20


def raster(kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "one channel":  # distances 0..9: the mean of a 3x3 window is often one of them
        a = np.zeros((H, W, 3), np.uint8)
        a[..., 1] = rng.integers(0, 10, (H, W))
    elif kind == "three levels":
        a = (rng.integers(0, 3, (H, W, 3)) * 60).astype(np.uint8)
    elif kind == "extremes":
        a = (rng.integers(0, 2, (H, W, 3)) * 255).astype(np.uint8)
    else:  # smooth, with flat boxes
        y, x = np.mgrid[:H, :W]
        a = np.stack([x + y, 2 * x, 3 * y], 2) + rng.integers(0, 4, (H, W, 3))
        a = np.clip(a, 0, 255).astype(np.uint8)
        a[10:30, 40:70] = 77
    return a


@pytest.mark.parametrize("window", [(3, 3), (5, 5), (9, 7), (3, 11), (11, 11)])
@pytest.mark.parametrize("kind", ["one channel", "three levels", "extremes", "smooth"])
def test_color_census_ties(gpu_context, kind, window):
    lb = raster(kind, 5)
    rb = np.roll(lb, -6, axis=1).copy()
    rb[:, -6:] = raster(kind, 6)[:, -6:]
    left, right = bgr_gray(lb), bgr_gray(rb)
    op = O.params(window_w=window[0], window_h=window[1], disparities=D, cost=0, lr_threshold=1.0)
    print("colour ties", kind, window, flush=True)
    want = O.compute_color(op, left, right, lb, rb, W, H, None, None)
    got = gpu_context.match_pair_color(to_sgm(op), left, right, lb, rb)
    assert_same(got, want, "colour ties %s %r" % (kind, window))
