"""Large host copies in pieces: sizes around the pieces, the rule's limit and
the number of threads, through a grid's export and a sky's upload."""
import math

import numpy as np
import pytest

import blacktracer_amd as bt
from blacktracer_amd import scene
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [7, 8, 9, 10])
def test_export(ctx, level):
    """Each array alone equals the arrays exported together."""
    hole = bt.BlackHole(0.9)
    g = bt.Grid(level, level, True, bt.Camera(1.2, 0.0, 6.0, black_hole=hole), hole, ctx=ctx)
    L = bt._lib.load()
    cel, steps = np.full((g.N, g.M, 2), 7.0), np.full((g.N, g.M), 7, np.int32)
    bt.check(L.bt_grid_export(g.handle, cel.ctypes.data_as(bt._lib.DP), None, None))
    bt.check(L.bt_grid_export(g.handle, None, steps.ctypes.data_as(bt._lib.I32P), None))
    assert np.array_equal(cel, g.cel) and np.array_equal(steps, g.steps)
    i, j = g.N // 3, g.M // 5
    th, ph, st = bt.trace_rays(bt.Camera(1.2, 0.0, 6.0, black_hole=hole),
                               np.array([i / (g.N - 1) * math.pi]), np.array([j / g.M * 2 * math.pi]), ctx=ctx)
    assert (g.cel[i, j, 0], g.cel[i, j, 1], g.steps[i, j]) == (th[0], ph[0], st[0])


@pytest.mark.parametrize("rows,cols", [(1024, 1365), (1025, 1366), (1, 1400001), (2049, 4097)])
def test_sky_upload(ctx, rows, cols):
    sky = np.random.default_rng(cols).integers(0, 256, (rows, cols, 3), dtype=np.uint8)
    sc = bt.Scene(scene.synthetic_stars(50, 3), sky, tree_level=3, ctx=ctx)
    assert np.array_equal(sc.table(), O.sum_table(sky))
