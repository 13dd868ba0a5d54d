"""The render pass where its kernels hand pixels to each other, against the
CPU oracle: star counts that leave pixels dark, to one lane, to chunks or (a
small frame of a dense sky) without chunk room; quads across phi = 2 pi and
of many bin rows; odd pixels (a star beyond the fast taps' magnitudes makes
every pixel one); frames at the edges of the 16 x 16 tiles and of the
workgroups' four-tile runs; skies narrower than a footprint, where the column
sums take their last branch; a column count that is no multiple of the lanes.

Bars of the frame tests: 1/255 per channel, at most 0.1% of pixels differing;
star light within 1e-4 relative (its sums are reassociated).
"""
import math

import numpy as np
import pytest

import blacktracer_amd as bt
from blacktracer_amd import scene as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

VIEW = (math.pi / 2, 0.0, 0.25 * math.pi / 4)


@pytest.fixture(scope="module")
def pose(ctx):
    bh = bt.BlackHole(0.999)
    cam = bt.Camera(math.pi / 2, 0.0, 5.0, black_hole=bh)
    return cam, bt.Grid(7, 1, True, cam, bh, ctx=ctx)


def _check(ctx, pose, stars, sky, W, H, flags, step=1, level=8):
    cam, g = pose
    sc = bt.Scene(stars, sky, tree_level=level, ctx=ctx)
    img, st = bt.render_frame(g, sc, bt.View(W, H, ctx=ctx), flags=flags, step=step, stages=True)
    tree, pos, mag = O.make_tree(stars, level)
    oimg, ost = O.frame(g.cel.astype(np.float32), g.MAXLEVEL, O.camera_view(*VIEW, W, H), cam.getParamArray(), tree,
                        level, pos, mag, O.sum_table(sky), star=flags.star, map=flags.map, lr=flags.lr, hor=flags.hor,
                        ver=flags.ver, offset=flags.offset, step=step, stages=True)
    assert np.array_equal(st["thphi"], ost["thphi"]) and np.array_equal(st["bh"], ost["bh"])
    nb = st["bh"] == 0
    assert np.array_equal(st["area"][nb], ost["area"][nb])
    if flags.star:
        assert np.allclose(st["star"], ost["star"], rtol=1e-4, atol=1e-3, equal_nan=True)
    d = np.abs(img.astype(np.int16) - oimg.astype(np.int16)).max(axis=-1)
    print(f"  {W}x{H} step {step}, {len(stars)} stars, sky {sky.shape[1]}: max {d.max()}, {(d > 0).mean():.2e} differ",
          flush=True)
    assert d.max() <= 1 and (d > 0).mean() <= 1e-3


@pytest.mark.parametrize("W,H,step,stars,offset", [
    (16, 16, 1, 300, 0.0),          # one tile
    (17, 15, 2, 300, 0.3),          # one pixel over, three of a splat's reach
    (33, 18, 1, 60000, 0.5),        # more chunks than the frame has room for
    (250, 141, 3, 0, 0.1),          # no star at all
    (250, 141, 1, 40, 2.9),         # nearly all dark, wide quads of few candidates
    (321, 180, 1, 40000, 1.7),      # quads across the seam, chunks of several hundreds
    (1031, 1024, 1, 3000, 0.2),     # four-tile workgroups, ragged on the right
])
def test_star_classes(ctx, pose, W, H, step, stars, offset):
    s4 = S.synthetic_stars(stars, seed=3 + stars)
    _check(ctx, pose, s4, S.synthetic_sky(256, seed=4), W, H, bt.RenderFlags(map=False, offset=offset), step=step)


@pytest.mark.parametrize("level", [1, 6, 10])
def test_star_tree_levels(ctx, pose, level):
    _check(ctx, pose, S.synthetic_stars(9000, seed=8), S.synthetic_sky(256, seed=4), 201, 119,
           bt.RenderFlags(map=False, offset=0.9), level=level)


def test_every_pixel_odd(ctx, pose):
    s4 = S.synthetic_stars(12000, seed=12)
    s4[17, 2] = -11.0               # beyond the fast taps' magnitudes
    _check(ctx, pose, s4, S.synthetic_sky(256, seed=4), 193, 110, bt.RenderFlags(map=False, offset=0.4))


@pytest.mark.parametrize("cols", [32, 63 * 2, 1024, 2050])
@pytest.mark.parametrize("W,H", [(97, 61), (640, 33)])
def test_sky_columns(ctx, pose, cols, W, H):
    sky = np.random.default_rng(cols).integers(0, 256, (cols // 2, cols, 3), dtype=np.uint8)
    _check(ctx, pose, S.synthetic_stars(10, seed=1), sky, W, H, bt.RenderFlags(star=False, offset=0.8))


def test_moving_camera_redshift(ctx):
    """A camera off its orbit takes the full redshift expression."""
    bh = bt.BlackHole(0.7)
    cam = bt.Camera(1.2, 0.0, 8.0, 0.3, math.sqrt(1 - 0.3 * 0.3 - 0.6 * 0.6), 0.6, black_hole=bh)
    g = bt.Grid(6, 1, True, cam, bh, ctx=ctx)
    _check(ctx, (cam, g), S.synthetic_stars(5000, seed=2), S.synthetic_sky(512, seed=6), 160, 90,
           bt.RenderFlags(offset=0.1))
