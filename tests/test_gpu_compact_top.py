"""Compact plan with penalties near the 16-bit bound and the true disparity at the
top of the range: verified pixels whose winner lies beside the pad cells of their
row, in every position of the range's end within a group of four cells.  Results
equal the resident plan's bit for bit."""
import numpy as np
import pytest

from pose_amd import sgm, synth
from tests.test_gpu_compact_lines import _params
from tests.test_gpu_esgm import esgm
from tests.test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu

# (D, paths, P1, P2): eight paths hold P2 up to 7679 in 16 bits, the line sweeps 9216
CASES = [(D, 8, 600, 7600) for D in (89, 90, 91, 92)] + [(D, 4, 900, 9216) for D in (57, 90, 127)] \
    + [(250, 8, 300, 7679), (341, 8, 600, 7600), (449, 4, 900, 9216)]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("below", [1, 2, 3])
def test_top_of_the_range_equals_resident(gpu_context, case, below):
    D, dirs, p1, p2 = CASES[case]
    w, h, shift = D + 90, 31, D - 1 - below
    rng = np.random.default_rng(D + below)
    left, _, _ = synth.stereo_pair(w, h, 8, 0, seed=D)
    left = np.array(left)
    right = rng.integers(0, 256, (h, w)).astype(np.uint8)
    right[:, :w - shift] = left[:, shift:]
    noise = rng.integers(-6, 7, (h, w))
    right = np.clip(right + noise, 0, 255).astype(np.uint8)
    p = _params(D, 0, dirs, p1=p1, p2=p2)
    want = gpu_context.match_pair(p, left, right)
    got, counts = esgm(gpu_context, p, left, right, rows=h, pool=1, what="top D %d" % D)
    assert counts["left"][1] > 0
    assert_same(got, want, "D %d" % D)
