"""Reading results back: bodies and manifolds of one world and of every world
of a batch, in order, in reverse, after edits and destroyed neighbours, more
than one piece of pinned memory at a time, against a world of the same scene
stepped and read alone."""
import ctypes

import numpy as np
import pytest

from helpers import bits_equal, first_diff

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0


def _worlds(ctx, specs):
    from resolve2d_amd.engine import GpuWorld, apply_scene
    out = []
    for ops in specs:
        w = GpuWorld(ctx)
        apply_scene(ops, w)
        out.append(w)
    return out


def _oracle(oracle, ops, steps):
    from resolve2d_amd.engine import apply_scene
    o = oracle.OracleWorld("f32")
    apply_scene(ops, o)
    for _ in range(steps):
        assert o.process(DT, 4, 4) == 0
    return o


@pytest.mark.parametrize("order", ["forward", "backward", "every third"])
def test_reading_a_batch(oracle, order):
    from resolve2d_amd import scenes
    from resolve2d_amd.solver import Context
    ctx = Context(0)
    specs = [scenes.batched_world(300 + k, n_min=2 + 3 * k, n_max=2 + 3 * k) for k in range(40)]
    ws = _worlds(ctx, specs)
    idx = {"forward": range(40), "backward": range(39, -1, -1), "every third": range(0, 40, 3)}[order]
    for rnd in range(2):
        ctx.process_batch_handles([w.handle for w in ws], DT, 4, 4, 2)
        gone = 5 if rnd else None
        if rnd:
            ws[gone].close()            # a neighbour that is no longer there
            ws[7].exclude(1, 2)         # an edit without a step
        for i in idx:
            if i == gone:
                continue
            o = _oracle(oracle, specs[i], 2 * (rnd + 1))
            a, b = ws[i].bodies(), o.bodies()
            assert bits_equal(a, b), (rnd, i, first_diff(a, b))
            if i != 7 or not rnd:
                ma, mb = ws[i].manifolds(), o.manifolds()
                assert ma.shape == mb.shape and bits_equal(ma, mb), (rnd, i)
            o.close()
    for i, w in enumerate(ws):
        if i != 5:
            w.close()
    ctx.close()


@pytest.mark.parametrize("n", [1, 3000, 30000])
def test_reading_pieces(n):
    """Manifolds in pieces of the caller's choice equal those read at once;
    bodies added on the device are read whole (masses and shapes too)."""
    from resolve2d_amd import _native as N
    from resolve2d_amd import scenes
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    ctx = Context(0)
    w = GpuWorld(ctx)
    apply_scene(scenes.mixed(n, seed=2, width=2.0 * n ** 0.5, height=n ** 0.5, ground_w=4.0 * n ** 0.5 + 8.0), w)
    for _ in range(3):
        assert w.process(DT, 4, 4) == 0
    whole = w.manifolds()
    count = ctypes.c_size_t()
    for cap in (0, 1, len(whole) // 2, len(whole) + 5):
        arr = (N.ManifoldState * max(cap, 1))()
        N.check(w.lib.r2d_get_manifolds(w.handle, arr, cap, ctypes.byref(count)), "r2d_get_manifolds")
        assert count.value == len(whole)
        got = np.frombuffer(arr, np.uint32).reshape(max(cap, 1), -1)[:min(cap, len(whole)), :2]
        assert (got == whole[:len(got), :2]).all()
    first = w.bodies()
    assert bits_equal(first, w.bodies()) and np.isfinite(first).all()
    w.close()
    ctx.close()
