"""Long narrow images, whose few long lines set the time of the sweeps: single planes
in the narrow wave shapes, not planes of pairs; sequential 32-bit sweeps where the
pairs' chain would be longer; widths past 65535.  Results equal the one-aggregate
schedule bit for bit, alone and in phase-major batches, and the choice is no slower
than that schedule."""
import time

import numpy as np
import pytest

from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu

CENSUS, ZNCC32 = 0, 4


def params(D, md=0, p2=120, dirs=8, sums=0, cost=CENSUS):
    return sgm.SgmParams(window_w=5, window_h=5, disparities=D, min_disparity=md, cost=cost, p1=10,
                         p2=p2, edge_scale=32, directions=dirs, aggregate_bytes=sums,
                         census_weight=500, ad_truncation=30, gradient_truncation=60, reserved=0,
                         uniqueness=0.03, lr_threshold=1.0)


def match(p, left, right, schedule):
    ctx = sgm.Context(0)
    try:
        ctx.sweeps(schedule)
        ctx.match_pair(p, left, right)
        ctx.set_profiling(True)
        runs = []
        for _ in range(3):
            ctx.profile()
            out = ctx.match_pair(p, left, right)
            runs.append({k: v["total_ms"] for k, v in
                         ctx.profile()["device_kernel_milliseconds"].items()})
        return out, runs[0], min(sum(v for k, v in r.items() if k.startswith("path")) for r in runs)
    finally:
        ctx.close()


def assert_equal(got, want):
    for k in ("checked", "dl", "dr"):
        assert np.array_equal(got[k].view(np.uint32), want[k].view(np.uint32)), k
    for k in ("reasons", "boundary"):
        assert np.array_equal(got[k], want[k]), k
    assert got["stats"] == want["stats"]


# every padded row that has a narrow shape, full and partly filled, wide and tall,
# uint8 and uint16 costs, 4 and 8 paths, in the caches and beyond them
CASES = [(700, 23, 65, 0, 120, 8, CENSUS), (900, 31, 128, -7, 150, 8, CENSUS),
         (29, 800, 190, 0, 120, 8, CENSUS), (1100, 40, 192, 0, 120, 4, CENSUS),
         (1300, 22, 250, 3, 150, 8, CENSUS), (31, 1000, 256, 0, 120, 8, CENSUS),
         (1500, 21, 300, 0, 120, 8, CENSUS), (1400, 24, 320, -11, 150, 8, CENSUS),
         (1600, 20, 384, 0, 120, 8, CENSUS), (25, 1300, 400, 0, 120, 8, CENSUS),
         (1700, 20, 448, 0, 150, 4, CENSUS), (1900, 20, 512, 0, 120, 8, CENSUS),
         (2100, 20, 600, 0, 120, 8, CENSUS), (2300, 20, 640, 0, 120, 8, CENSUS),
         (900, 31, 128, 0, 150, 8, ZNCC32), (1000, 30, 192, 0, 150, 8, ZNCC32),
         (1200, 25, 320, 0, 150, 8, ZNCC32), (1900, 20, 512, 0, 150, 4, ZNCC32),
         (9000, 90, 128, 0, 120, 8, CENSUS), (6000, 70, 256, 0, 120, 8, CENSUS),
         (8000, 50, 320, 0, 150, 8, CENSUS), (60, 5000, 384, 0, 120, 8, CENSUS),
         (70000, 12, 500, 0, 24, 8, CENSUS)]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_long_images_equal_the_aggregate(case):
    w, h, D, md, p2, dirs, cost = CASES[case]
    p = params(D, md, p2, dirs, 0, cost)
    left, right, _ = synth.stereo_pair(w, h, min(D, w - 2), md, seed=300 + case)
    print("long", CASES[case], flush=True)
    got, ran, _ = match(p, left, right, "auto")
    assert "path_excess" in ran
    want, _, _ = match(p, left, right, "sequential")
    assert_equal(got, want)


@pytest.mark.parametrize("w,h,D,sums", [(12000, 40, 128, 2), (12000, 40, 256, 2), (40, 12000, 256, 2),
                                        (9000, 40, 320, 2), (9000, 40, 512, 2), (20000, 20, 192, 4),
                                        (20000, 15, 256, 4), (1200, 30, 256, 4),
                                        (16000, 106, 256, 4)])
def test_long_images_take_no_longer_than_the_aggregate(w, h, D, sums):
    p = params(D, sums=sums)
    left, right, _ = synth.stereo_pair(w, h, min(D, w - 2), 0, seed=D)
    got, ran, auto_ms = match(p, left, right, "auto")
    want, _, sequential_ms = match(p, left, right, "sequential")
    print("long", w, h, D, sums, "path ms", auto_ms, "sequential", sequential_ms, flush=True)
    assert_equal(got, want)
    # (where the sequential sweeps are the choice, the two are the same work)
    assert auto_ms <= (1.1 if "path_excess" not in ran else 1.0) * sequential_ms


@pytest.mark.parametrize("graph", [False, True])
def test_long_images_in_a_batch(graph):
    # one lane group of two narrow shapes, and one narrow shape of two ordinary ones
    sizes = [(900, 30, 128), (1000, 25, 192), (30, 1100, 250), (1500, 20, 300), (1600, 22, 500)]
    ctx = sgm.Context(0)
    try:
        records, buffers, want = [], [], []
        for i, (w, h, D) in enumerate(sizes):
            left, right, _ = synth.stereo_pair(w, h, min(D, w - 2), 0, seed=60 + i)
            fresh = sgm.Context(0)
            fresh.sweeps("sequential")
            want.append(fresh.match_pair(params(D), left, right))
            fresh.close()
            n = w * h
            b = [ctx.alloc(n).upload(left), ctx.alloc(n).upload(right), ctx.alloc(4 * n),
                 ctx.alloc(4 * n), ctx.alloc(4 * n), ctx.alloc(128)]
            buffers.append(b)
            records.append(sgm.SgmPair(width=w, height=h, disparities=D, min_disparity=0,
                                       left=b[0].ptr, right=b[1].ptr, checked=b[2].ptr, dl=b[3].ptr,
                                       dr=b[4].ptr, stats=b[5].ptr))
        batch = sgm.DeviceBatch(ctx, params(64), records, graph=graph, phased=True)
        assert batch.describe()["sweeps"] == "planes"
        for _ in range(3):
            print("long batch", graph, flush=True)
            batch.run()
            ctx.synchronize()
            for b, r in zip(buffers, want):
                for buf, k in zip(b[2:5], ("checked", "dl", "dr")):
                    assert np.array_equal(buf.download(np.uint32, r[k].size), r[k].view(np.uint32)), k
        batch.close()
        for b in buffers:
            for x in b:
                x.free()
    finally:
        ctx.close()


def test_ordinary_pairs_beside_a_long_one_keep_their_shape():
    # the narrow waves of one long image are not taken to the others, which take
    # no longer with it beside them than both by themselves
    sizes = [(4000, 60, 128), (640, 480, 128), (640, 480, 128)]

    def run(sizes):
        ctx = sgm.Context(0)
        try:
            records = []
            for i, (w, h, D) in enumerate(sizes):
                left, right, _ = synth.stereo_pair(w, h, D, 0, seed=80 + i)
                n = w * h
                b = [ctx.alloc(n).upload(left), ctx.alloc(n).upload(right), ctx.alloc(4 * n)]
                records.append(sgm.SgmPair(width=w, height=h, disparities=D, min_disparity=0,
                                           left=b[0].ptr, right=b[1].ptr, checked=b[2].ptr))
            batch = sgm.DeviceBatch(ctx, params(64), records, phased=True)
            least = 1e9
            for _ in range(8):
                ctx.synchronize()
                start = time.perf_counter()
                batch.run()
                ctx.synchronize()
                least = min(least, time.perf_counter() - start)
            batch.close()
            return 1e3 * least
        finally:
            ctx.close()

    together, long, others = run(sizes), run(sizes[:1]), run(sizes[1:])
    print("long batch ms", together, "long", long, "others", others, flush=True)
    assert together <= 1.05 * (long + others)
