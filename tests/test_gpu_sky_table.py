"""The summed sky table at sizes that leave remainders of its blocks and row
batches, bit for bit with the CPU oracle (which sums each column in order)."""
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
