"""Grids whose first levels are traced ahead: the same grid whichever level
that is, and the statistics of the rays that its blocks asked for alone.

A single grid traces a finer lattice ahead than the same grid in a batch of
many, so each must equal the other bit for bit; the counts must equal those of
a ray batch over exactly the traced directions.
"""
import math

import numpy as np
import pytest

import blacktracer_amd as bt

pytestmark = pytest.mark.gpu

COUNTS = ("rays", "integrated", "attempts", "attempts_fp64", "newton", "golden", "fallback_rays")


def traced_directions(g):
    """Directions of the rays a build traces: every present point but the
    copies along the pole rows at the start level's spacing."""
    present = g.cel[..., 0] != -2
    gap0 = 1 << (g.MAXLEVEL - g.STARTLVL)
    for row in (0, g.N - 1) if g.equafactor else (0,):
        present[row, gap0::gap0] = False
    i, j = np.nonzero(present)
    return i / (g.N - 1) * math.pi / (2 - g.equafactor), j / g.M * (2 * math.pi)


def camera(k):
    hole = bt.BlackHole(0.0 if k == 3 else 0.999 - 0.07 * k)
    return bt.Camera(math.pi / 2 - 0.1 * k, 0.0, 4.0 + k, black_hole=hole), hole


FP64, MIXED = {}, {"precision": bt.BT_PREC_MIXED}


@pytest.mark.parametrize("level,start,angle,thresh,prm", [
    (1, 1, True, 0.015, FP64), (2, 1, False, 0.015, FP64), (5, 5, True, 0.015, FP64), (8, 1, True, 0.015, FP64),
    (8, 3, False, 0.015, FP64), (9, 6, True, 0.015, FP64), (8, 2, True, 1e9, FP64), (10, 1, False, 0.1, FP64),
    (1, 1, False, 0.015, MIXED), (8, 1, True, 0.015, MIXED), (8, 4, False, 0.015, MIXED), (9, 1, True, 0.1, MIXED),
    (6, 2, True, 0.015, {**MIXED, "eps": 1e-8}), (7, 1, True, 0.015, {**MIXED, "apriori_capture": 0, "r_capture_factor": 1.01}),
    (7, 1, True, 0.015, {**FP64, "max_steps": 60})])
def test_same_grid_and_counts(ctx, level, start, angle, thresh, prm):
    n = 3 if level > 9 else 36
    cams, holes = zip(*[camera(k % 5) for k in range(n)])
    prm = bt.IntegParams(**prm)
    print(f"batch of {n} Grid({level},{start},angle={angle}) thresh={thresh} precision={prm.precision}", flush=True)
    batch, stats = bt.Grid.build_batch(cams, holes, [level] * n, [start] * n, angle=angle, params=prm,
                                       refine_thresh=thresh, fix_tvertices=False, ctx=ctx)
    total = dict.fromkeys(COUNTS, 0)
    for k in range(min(n, 5)):
        g = bt.Grid(level, start, angle, cams[k], holes[k], params=prm, refine_thresh=thresh, fix_tvertices=False,
                    ctx=ctx)
        for h in batch[k::5]:
            assert g.rays_traced == h.rays_traced
            assert np.array_equal(g.cel, h.cel) and np.array_equal(g.steps, h.steps)
            assert np.array_equal(g.levels, h.levels)
        assert not g.steps[g.cel[..., 0] == -2].any()
        th, ph = traced_directions(g)
        assert th.size == g.rays_traced
        *_, want = bt.trace_rays(cams[k], th, ph, params=prm, ctx=ctx, return_stats=True)
        assert {c: g.stats()[c] for c in COUNTS} == {c: want[c] for c in COUNTS}
        for c in COUNTS:
            total[c] += want[c] * len(batch[k::5])
    assert {c: stats[c] for c in COUNTS} == total
    for h in batch:
        h.close()


def test_uniform_batch_counts(ctx):
    """A batch whose grids all start at their last level, and one that mixes
    such grids with adaptive ones, against the single grids."""
    for levels, starts in (([7, 6, 7], [7, 6, 7]), ([7, 7, 6], [7, 2, 6])):
        cams, holes = zip(*[camera(k) for k in range(3)])
        print(f"batch of levels {levels} from {starts}", flush=True)
        batch, stats = bt.Grid.build_batch(cams, holes, levels, starts, ctx=ctx)
        total = dict.fromkeys(COUNTS, 0)
        for k, h in enumerate(batch):
            g = bt.Grid(levels[k], starts[k], True, cams[k], holes[k], ctx=ctx)
            assert g.rays_traced == h.rays_traced and g.rays_traced == g.stats()["rays"]
            assert np.array_equal(g.cel, h.cel) and np.array_equal(g.steps, h.steps)
            for c in COUNTS:
                total[c] += g.stats()[c]
        assert {c: stats[c] for c in COUNTS} == total


@pytest.mark.parametrize("prm", [FP64, MIXED])
def test_threshold_beyond_every_jump(ctx, prm):
    """Thresholds above the largest distance of two grid values, infinite and
    no number: the grid of the largest threshold below it, and no finer
    lattice traced for it than the blocks that always refine ask for."""
    cam, hole = camera(1)
    prm = bt.IntegParams(**prm)
    name = "ic_split" if prm.precision == bt.BT_PREC_MIXED else "ic_capture_f64"

    def build(level, start, thresh):
        print(f"Grid({level},{start}) thresh={thresh} precision={prm.precision}", flush=True)
        g = bt.Grid(level, start, True, cam, hole, params=prm, refine_thresh=thresh, ctx=ctx)
        return g, (g.cel, g.steps, g.levels, g.rays_traced)

    for level, start in ((5, 1), (9, 2), (9, 6), (9, 7), (8, 8)):
        _, want = build(level, start, 70.5)
        for thresh in (71.0, 1e300, math.inf, math.nan):
            _, got = build(level, start, thresh)
            assert all(np.array_equal(a, b) for a, b in zip(got, want))
        assert want[2].max() == max(start, min(level, 6))
    capture = []
    ctx.timing(True)
    try:
        for thresh in (70.5, 71.0):
            build(12, 6, thresh)   # buffers
            ctx.reset_timers()
            build(12, 6, thresh)
            capture.append(ctx.timer(name)[1])
    finally:
        ctx.timing(False)
    print(f"capture test {capture} ms", flush=True)
    assert capture[1] < 0.5 * capture[0]
