"""Ray batches around the sizes where the launch shape changes (one wave,
three quarters of a wave, one and three waves per SIMD, one ray per resident
lane): each equals the same rays of one larger batch bit for bit."""
import math

import numpy as np
import pytest

import blacktracer_amd as bt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [bt.BT_PREC_FP64, bt.BT_PREC_MIXED])
def test_prefixes(ctx, precision):
    cam = bt.Camera(1.3, 0.0, 6.0, black_hole=bt.BlackHole(0.9))
    rng = np.random.default_rng(11)
    n = 140001
    th, ph = np.arccos(1 - 2 * rng.random(n)), 2 * math.pi * rng.random(n)
    prm = bt.IntegParams(precision)
    whole = bt.trace_rays(cam, th, ph, params=prm, ctx=ctx)
    for k in (1, 63, 64, 65, 129, 500, 65535, 65536, 65537, 131072, 131073):
        print(f"{k} rays, precision {precision}", flush=True)
        part = bt.trace_rays(cam, th[:k], ph[:k], params=prm, ctx=ctx)
        assert all(np.array_equal(a, b[:k]) for a, b in zip(part, whole))


def test_mixed_reservations(ctx):
    """The FP32 bulk's and the critical rays' reservations change at three
    quarters of a wave and at three waves per SIMD."""
    cam = bt.Camera(1.3, 0.0, 6.0, black_hole=bt.BlackHole(0.9))
    rng = np.random.default_rng(12)
    n = 350001
    th, ph = np.arccos(1 - 2 * rng.random(n)), 2 * math.pi * rng.random(n)
    prm = bt.IntegParams(bt.BT_PREC_MIXED)
    whole = bt.trace_rays(cam, th, ph, params=prm, ctx=ctx)
    for k in (49151, 49152, 49153, 196607, 196608, 196609):
        print(f"{k} rays", flush=True)
        part = bt.trace_rays(cam, th[:k], ph[:k], params=prm, ctx=ctx)
        assert all(np.array_equal(a, b[:k]) for a, b in zip(part, whole))
