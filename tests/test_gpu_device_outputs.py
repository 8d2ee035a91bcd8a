"""Disparity outputs of the device entry points: written in place where the
caller's map stands alone, copied at the end where it shares memory with another
buffer of the call or is not float-aligned; the results are the same."""
import numpy as np
import pytest

from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu

W, H, D = 140, 90, 48
N = W * H


def params():
    return sgm.SgmParams(window_w=9, window_h=7, disparities=D, min_disparity=0, cost=0, p1=10,
                         p2=120, edge_scale=32, directions=8, aggregate_bytes=0,
                         census_weight=500, ad_truncation=30, gradient_truncation=60, reserved=0,
                         uniqueness=0.03, lr_threshold=1.0)


@pytest.mark.parametrize("entry", ["match_pair_device", "match_pair_device_noalloc"])
@pytest.mark.parametrize("layout", ["apart", "dl is dr", "dl is checked", "dr overlaps dl",
                                    "dl misaligned", "dl on the left image"])
def test_disparity_outputs(gpu_context, entry, layout):
    ctx = gpu_context
    left, right, _ = synth.stereo_pair(W, H, D, 0, seed=31)
    want = ctx.match_pair(params(), left, right)
    arena = ctx.alloc(16 * N)  # the maps lie in one allocation
    inputs = ctx.alloc(5 * N)
    inputs.upload(left)
    dright, stats = ctx.alloc(N).upload(right), ctx.alloc(128)
    checked, dl, dr = arena.ptr, arena.ptr + 4 * N, arena.ptr + 8 * N
    if layout == "dl is dr":
        dr = dl
    elif layout == "dl is checked":
        dl = checked
    elif layout == "dr overlaps dl":
        dr = dl + 2 * N
    elif layout == "dl misaligned":
        dl = arena.ptr + 12 * N - 2 * N + 2
        dr = arena.ptr + 4 * N
    elif layout == "dl on the left image":
        dl = inputs.ptr
    print("device outputs", entry, layout, flush=True)
    getattr(ctx, entry)(params(), inputs.ptr, dright.ptr, W, H, checked, d_dl=dl, d_dr=dr,
                        d_stats=stats.ptr)
    ctx.synchronize()

    def read(base, ptr):
        raw = base.download(np.uint8, base.nbytes)
        off = ptr - base.ptr
        return raw[off:off + 4 * N].copy().view(np.uint32)

    bits = {k: want[k].view(np.uint32) for k in ("checked", "dl", "dr")}
    # the copies come last, dl before dr: a later output covers an earlier one
    if layout != "dl is checked":
        assert np.array_equal(read(arena, checked), bits["checked"])
    if layout == "dr overlaps dl":
        assert np.array_equal(read(arena, dl)[:N // 2], bits["dl"][:N // 2])
    elif layout != "dl is dr":
        assert np.array_equal(read(inputs if layout == "dl on the left image" else arena, dl),
                              bits["dl"])
    assert np.array_equal(read(arena, dr), bits["dr"])
    assert stats.download(np.int64, 16)[10] == want["stats"]["valid"]
    for b in (arena, inputs, dright, stats):
        b.free()
