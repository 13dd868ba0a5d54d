"""Native objects are freed after those made from them, in whatever order
their Python objects are closed or finalised."""
import gc
import itertools

import numpy as np
import pytest

import blacktracer_amd as bt

PARENTS = {"grid": {"context"}, "scene": {"context"}, "view": {"context"}, "trails": {"context"},
           "server": {"context", "scene"}, "device": {"context"}, "context": set()}


class Library:
    """Stands in for the native library: hands out handles, records frees."""

    def __init__(self):
        self.freed = []
        self.handles = 0

    def __getattr__(self, name):
        def call(*args):
            if name.endswith(("_create", "_alloc", "_build")):
                self.handles += 1
                args[-1]._obj.value = self.handles
            elif name.endswith(("_free", "_destroy")):
                assert args[0], f"{name} of a null handle"
                self.freed.append(name.split("_")[1])
            return 0
        return call


def objects(monkeypatch):
    lib = Library()
    monkeypatch.setattr(bt._lib, "load", lambda: lib)
    ctx = bt.Context(0)
    hole = bt.BlackHole(0.9)
    scene = bt.Scene(np.zeros((1, 4), np.float32), np.zeros((1, 2, 3), np.uint8), ctx=ctx)
    made = [ctx, scene, bt.Server(scene, ctx=ctx), bt.Trails(scene, 16, 9, ctx=ctx),
            bt.Grid(1, 1, True, bt.Camera(1.0, 0.0, 5.0, black_hole=hole), hole, ctx=ctx), bt.View(16, 9, ctx=ctx),
            ctx.alloc(64)]
    return lib, made


def check(freed):
    assert sorted(freed) == sorted(PARENTS)
    for k, name in enumerate(freed):
        assert not PARENTS[name] & set(freed[:k]), f"{name} freed after its parent: {freed}"


@pytest.mark.parametrize("order", list(itertools.permutations(range(4))))
def test_closed_in_any_order(monkeypatch, order):
    lib, made = objects(monkeypatch)
    for k in order + (4, 5, 6):
        made[k].close()
        made[k].close()
    check(lib.freed)


@pytest.mark.parametrize("turn", range(7))
def test_garbage_in_any_order(monkeypatch, turn):
    lib, made = objects(monkeypatch)
    ring = made[turn:] + made[:turn]
    for a, b in zip(ring, ring[1:] + ring[:1]):
        a.next = b
    del made, ring, a, b
    gc.collect()
    check(lib.freed)
