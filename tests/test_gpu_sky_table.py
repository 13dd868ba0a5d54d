"""The summed sky table at sizes that leave remainders of its blocks and row
batches, bit for bit with the CPU oracle (which sums each column in order)."""
import ctypes as C

import numpy as np
import pytest

import blacktracer_amd as bt
from blacktracer_amd import scene
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 64), (16, 65), (17, 63), (31, 130), (33, 64), (65, 1), (100, 199)])
def test_table_sizes(ctx, rows, cols):
    sky = np.random.default_rng(rows * 1000 + cols).integers(0, 256, (rows, cols, 3), dtype=np.uint8)
    print(f"sky {rows}x{cols}", flush=True)
    sc = bt.Scene(scene.synthetic_stars(50, 3), sky, tree_level=3, ctx=ctx)
    assert np.array_equal(sc.table(), O.sum_table(sky))


def test_more_pixels_than_an_index_holds(ctx):
    """Refused before the image is read."""
    L, sky, stars, out = bt._lib.load(), np.zeros(3, np.uint8), scene.synthetic_stars(1, 3), C.c_void_p()
    for rows, cols in ((46341, 46341), (1 << 30, 2), (2147483647, 2147483647)):
        with pytest.raises(bt.BtError):
            bt.check(L.bt_scene_create(ctx.handle, stars.ctypes.data_as(bt._lib.FP), 1, 3,
                                       sky.ctypes.data_as(bt._lib.U8P), rows, cols, C.byref(out)))
