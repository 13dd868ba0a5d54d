"""Large host copies in pieces: sizes around the pieces, the rule's limit and
the number of threads, through a grid's export and a sky's upload."""
import ctypes as C
import math

import numpy as np
import pytest
import torch

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


@pytest.mark.parametrize("level,angle", [(7, True), (9, False), (10, True)])
def test_export_equals_pinned(ctx, level, angle):
    """Every element of every array, alone and together, against an export
    into pinned memory, which the runtime copies by itself."""
    hole = bt.BlackHole(0.9)
    g = bt.Grid(level, 1, angle, bt.Camera(1.2, 0.0, 6.0, black_hole=hole), hole, ctx=ctx)
    L = bt._lib.load()
    kinds = (("cel", np.float64, bt._lib.DP), ("steps", np.int32, bt._lib.I32P),
             ("levels", np.int8, bt._lib.I8P))
    n = g.N * g.M
    want = []
    for k, (name, dtype, ptr) in enumerate(kinds):
        pinned = torch.full((n * (2 if k == 0 else 1),), 7, dtype=getattr(torch, np.dtype(dtype).name), pin_memory=True)
        args = [None] * 3
        args[k] = C.cast(pinned.data_ptr(), ptr)
        bt.check(L.bt_grid_export(g.handle, *args))
        want.append(pinned.numpy().copy())
        alone = np.full(pinned.numel(), 7, dtype)
        args[k] = alone.ctypes.data_as(ptr)
        bt.check(L.bt_grid_export(g.handle, *args))
        assert np.array_equal(alone, want[k]), f"{name} alone"
    together = [np.full(w.size, 7, w.dtype) for w in want]
    bt.check(L.bt_grid_export(g.handle, *[a.ctypes.data_as(ptr) for a, (_, _, ptr) in zip(together, kinds)]))
    for a, w, (name, _, _) in zip(together, want, kinds):
        assert np.array_equal(a, w), name
    for a, w in zip((g.cel, g.steps, g.levels), want):
        assert np.array_equal(a.ravel(), w)


def test_sky_upload_from_pinned(ctx):
    sky = torch.randint(0, 256, (1025, 1367, 3), dtype=torch.uint8).pin_memory().numpy()
    sc = bt.Scene(scene.synthetic_stars(50, 3), sky, tree_level=3, ctx=ctx)
    assert np.array_equal(sc.table(), O.sum_table(sky))


@pytest.mark.parametrize("rows,cols", [(1024, 1365), (1025, 1366), (1, 1400001), (2049, 4097)])
def test_sky_upload(ctx, rows, cols):
    sky = np.random.default_rng(cols).integers(0, 256, (rows, cols, 3), dtype=np.uint8)
    sc = bt.Scene(scene.synthetic_stars(50, 3), sky, tree_level=3, ctx=ctx)
    assert np.array_equal(sc.table(), O.sum_table(sky))
