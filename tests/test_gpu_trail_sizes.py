"""Trails and diffraction at the edges of their kernels against the CPU
oracle: a one-texel sprite whose window is the whole row, frames that are no
multiple of a tile, sprites across the frame's sides, more rows in reach of a
tile than one batch takes, the smallest and largest star tree.

Bars as in the sequence test: trails and summed light within 1e-4 relative,
frames within 1/255 per channel on all but 0.1% of the pixels (at least one
pixel).
"""
import math

import numpy as np
import pytest

import blacktracer_amd as bt
from blacktracer_amd import scene
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def world(ctx):
    hole = bt.BlackHole(0.999)
    cam = bt.Camera(math.pi / 2, 0.0, 5.0, black_hole=hole)
    return dict(cam=cam, grid=bt.Grid(8, 1, True, cam, hole, ctx=ctx))


@pytest.mark.parametrize("W,H,stars,level", [
    (16, 9, 20000, 8), (50, 31, 20000, 1), (203, 97, 30000, 10), (336, 40, 30000, 8), (4100, 280, 4000, 8)])
def test_sizes(ctx, world, W, H, stars, level):
    fs = W // 16
    y, x = np.mgrid[0:fs, 0:fs]
    sprite = np.stack([(37 * x + 11 * y) % 256, (5 * x * y + 90) % 256, np.full_like(x, 130)], -1).astype(np.uint8)
    stars = scene.synthetic_stars(stars, 17)
    sky = scene.synthetic_sky(256, seed=4)
    sc = bt.Scene(stars, sky, tree_level=level, ctx=ctx)
    tree, pos, mag = O.make_tree(stars, level)
    T, OT = bt.Trails(sc, W, H, diffraction=sprite, ctx=ctx), O.Trails(pos.shape[0], W, H, sprite)
    view = bt.View(W, H, ctx=ctx)
    oview = O.camera_view(math.pi / 2, 0.0, 0.25 * math.pi / 4, W, H)
    gridf, cam7 = world["grid"].cel.astype(np.float32), world["cam"].getParamArray()
    for k in range(2):
        off = k * 6 * math.pi / W
        print(f"{W}x{H} frame {k}", flush=True)
        img, st = T.render(world["grid"], sc, view, flags=bt.RenderFlags(offset=off), stages=True)
        oimg, olight, otrail = OT.frame(gridf, world["grid"].MAXLEVEL, oview, cam7, tree, level, pos, mag,
                                        O.sum_table(sky), offset=off)
        assert np.allclose(st["trail"], otrail, rtol=1e-4, atol=1e-3)
        assert np.allclose(st["star"], olight, rtol=1e-4, atol=1e-3, equal_nan=True)
        d = np.abs(img.astype(np.int16) - oimg.astype(np.int16)).max(axis=-1)
        assert d.max() <= 1 and (d > 0).sum() <= max(1, 1e-3 * W * H)
    T.close()
    OT.close()


@pytest.mark.parametrize("a,theta,r,W,H,count,least", [
    (0.3296, 1.42613, 6.5869, 1000, 560, 20000, 1),        # a handful beyond the slots
    (0.3634, 2.82043, 6.8094, 1976, 1111, 54075, 10000)])  # stars with hundreds of images
def test_more_images_than_a_star_keeps(ctx, a, theta, r, W, H, count, least):
    """Stars with more than 32 images in a frame keep the first in pixel order,
    as the oracle's do, in every run."""
    hole = bt.BlackHole(a)
    cam = bt.Camera(theta, 0.0, r, black_hole=hole)
    grid = bt.Grid(8, 1, True, cam, hole, ctx=ctx)
    stars = scene.synthetic_stars(count, 5)
    sky = np.zeros((16, 32, 3), np.uint8)
    sc = bt.Scene(stars, sky, tree_level=8, ctx=ctx)
    tree, pos, mag = O.make_tree(stars, 8)
    T, OT = bt.Trails(sc, W, H, ctx=ctx), O.Trails(pos.shape[0], W, H, None)
    view = bt.View(W, H, ctx=ctx)
    oview = O.camera_view(math.pi / 2, 0.0, 0.25 * math.pi / 4, W, H)
    gridf, table = grid.cel.astype(np.float32), O.sum_table(sky)
    dropped, want = 0, []
    for k in range(3):
        off = 0.3 + k * 3.0 / W
        print(f"frame {k}", flush=True)
        img, st = T.render(grid, sc, view, flags=bt.RenderFlags(offset=off), stages=True)
        _, olight, otrail = OT.frame(gridf, 8, oview, cam.getParamArray(), tree, 8, pos, mag, table, offset=off)
        assert np.allclose(st["trail"], otrail, rtol=1e-4, atol=1e-3)
        assert np.allclose(st["star"], olight, rtol=1e-4, atol=1e-3, equal_nan=True)
        dropped += T.stats()["dropped"]
        want.append((img, st["trail"]))
    print(f"{dropped} images dropped", flush=True)
    assert dropped >= least
    for run in range(4):
        T.reset()
        for k in range(3):
            img, st = T.render(grid, sc, view, flags=bt.RenderFlags(offset=0.3 + k * 3.0 / W), stages=True)
            assert np.array_equal(img, want[k][0]) and np.array_equal(st["trail"], want[k][1])
    T.close()
    OT.close()


def test_light_without_bound(ctx, world):
    """Stars bright enough for infinite light: what their sprite window does
    not cover keeps its light."""
    W, H = 160, 90
    sprite = np.full((W // 16, W // 16, 3), (0, 60, 255), np.uint8)
    stars = scene.synthetic_stars(20000, 17)
    stars[::3000, 2] = -120.0
    sky = scene.synthetic_sky(256, seed=4)
    sc = bt.Scene(stars, sky, tree_level=8, ctx=ctx)
    tree, pos, mag = O.make_tree(stars, 8)
    T, OT = bt.Trails(sc, W, H, diffraction=sprite, ctx=ctx), O.Trails(pos.shape[0], W, H, sprite)
    print("frame with infinite light", flush=True)
    img, st = T.render(world["grid"], sc, bt.View(W, H, ctx=ctx), stages=True)
    oimg, olight, _ = OT.frame(world["grid"].cel.astype(np.float32), world["grid"].MAXLEVEL,
                               O.camera_view(math.pi / 2, 0.0, 0.25 * math.pi / 4, W, H),
                               world["cam"].getParamArray(), tree, 8, pos, mag, O.sum_table(sky))
    assert not np.isfinite(olight).all() and np.isfinite(olight).mean() > 0.5
    assert np.allclose(st["star"], olight, rtol=1e-4, atol=1e-3, equal_nan=True)
    T.close()
    OT.close()
