"""Cost phase of batched runs without the fused census cost: rows of several pairs of
different sizes at once, as a grid of their own (phase-major) or as queue items; the
results are those of the pairs one by one."""
import time

import numpy as np
import pytest

from pose_amd import sgm, synth

pytestmark = pytest.mark.gpu


def params(cost, window=(7, 7), sums=0, dirs=4):
    return sgm.SgmParams(window_w=window[0], window_h=window[1], disparities=64, min_disparity=0,
                         cost=cost, p1=10, p2=96, edge_scale=32, directions=dirs,
                         aggregate_bytes=sums, census_weight=500, ad_truncation=30,
                         gradient_truncation=60, reserved=0, uniqueness=0.03, lr_threshold=1.0)


def records_of(ctx, sizes):
    records, buffers, images = [], [], []
    for i, (w, h, D, md) in enumerate(sizes):
        left, right, _ = synth.stereo_pair(w, h, max(3, min(D, w - 2)), md, seed=70 + i)
        n = w * h
        b = [ctx.alloc(n).upload(left), ctx.alloc(n).upload(right), ctx.alloc(4 * n),
             ctx.alloc(4 * n), ctx.alloc(4 * n), ctx.alloc(128)]
        buffers.append(b)
        images.append((left, right))
        records.append(sgm.SgmPair(width=w, height=h, disparities=D, min_disparity=md,
                                   left=b[0].ptr, right=b[1].ptr, checked=b[2].ptr, dl=b[3].ptr,
                                   dr=b[4].ptr, stats=b[5].ptr))
    return records, buffers, images


# one and two descriptor words, 8- and 16-bit volumes, 32-bit sums
@pytest.mark.parametrize("phased,graph", [(True, False), (True, True), (False, False)])
@pytest.mark.parametrize("cost,window,sums", [(0, (11, 11), 0), (0, (7, 7), 4), (1, (7, 7), 0),
                                              (1, (9, 9), 4), (2, (9, 7), 0), (3, (5, 5), 0),
                                              (3, (7, 7), 4), (4, (7, 7), 0)])
def test_costs_of_a_batch_match_single_pairs(cost, window, sums, phased, graph):
    # the images' last rows, rows narrower than a block, ranges of one quad and of many
    sizes = [(61, 47, 5, 0), (130, 13, 64, -7), (17, 90, 33, 3), (205, 31, 300, -20), (13, 13, 3, 0)]
    p = params(cost, window, sums)
    ctx = sgm.Context(0)
    try:
        records, buffers, images = records_of(ctx, sizes)
        want = []
        for (w, h, D, md), (left, right) in zip(sizes, images):
            q = params(cost, window, sums)
            q.disparities, q.min_disparity = D, md
            want.append(ctx.match_pair(q, left, right))
        batch = sgm.DeviceBatch(ctx, p, records, graph=graph, phased=phased)
        for _ in range(3):
            print("batch cost", cost, window, sums, phased, graph, flush=True)
            batch.run()
            ctx.synchronize()
            for b, r in zip(buffers, want):
                for buf, k in zip(b[2:5], ("checked", "dl", "dr")):
                    assert np.array_equal(buf.download(np.uint32, r[k].size), r[k].ravel().view(np.uint32)), k
        batch.close()
    finally:
        ctx.close()


def test_costs_of_many_pairs():
    # more rows than four to a wave: items of four rows, the last of an image shorter
    sizes = [(24, 43 + i % 5, 9, 0) for i in range(400)]
    ctx = sgm.Context(0)
    try:
        records, buffers, images = records_of(ctx, sizes)
        print("batch cost", len(sizes), flush=True)
        batch = sgm.DeviceBatch(ctx, params(1), records, phased=False)
        batch.run()
        ctx.synchronize()
        for (w, h, D, md), b, (left, right) in zip(sizes, buffers, images):
            q = params(1)
            q.disparities = D
            r = ctx.match_pair(q, left, right)
            for buf, k in zip(b[2:5], ("checked", "dl", "dr")):
                assert np.array_equal(buf.download(np.uint32, w * h), r[k].ravel().view(np.uint32)), k
        batch.close()
    finally:
        ctx.close()


def test_costs_of_a_few_pairs_fill_the_chip():
    # A phase-major run has the sweeps of the single pairs, several to a launch: its
    # costs must not make it slower than the pairs one by one.
    sizes = [(321, 152, 493, -19), (47, 1055, 448, 13), (324, 121, 256, 0), (236, 236, 320, 14)]
    ctx = sgm.Context(0)
    try:
        ctx.sweeps("sequential")
        records, buffers, _ = records_of(ctx, sizes)
        batch = sgm.DeviceBatch(ctx, params(1), records, phased=True)

        def pairs():
            for (w, h, D, md), b in zip(sizes, buffers):
                q = params(1)
                q.disparities, q.min_disparity = D, md
                ctx.match_pair_device(q, b[0].ptr, b[1].ptr, w, h, b[2].ptr, d_dl=b[3].ptr,
                                      d_dr=b[4].ptr)

        def best(run):
            least = 1e9
            for _ in range(8):
                ctx.synchronize()
                start = time.perf_counter()
                run()
                ctx.synchronize()
                least = min(least, time.perf_counter() - start)
            return 1e3 * least

        pairs(), batch.run()
        batch_ms, pairs_ms = best(batch.run), best(pairs)
        print("batch cost", "ms", batch_ms, "single pairs", pairs_ms, flush=True)
        assert batch_ms <= 1.25 * pairs_ms
        batch.close()
    finally:
        ctx.close()
