"""The step scratch where its first estimate or the device's memory is too
small: arrays that grow within a call, programs of fewer iterations.  Bit for
bit against the oracle."""
import pytest

from helpers import bits_equal, first_diff
from test_gpu_programs import _heap, _links
from test_rules import _room, rule

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0


def _same(g, o, where):
    a, b = g.bodies(), o.bodies()
    assert bits_equal(a, b), (where, first_diff(a, b))
    mg, mo = g.manifolds(), o.manifolds()
    assert mg.shape == mo.shape and bits_equal(mg, mo), (where, first_diff(mg, mo))


@pytest.mark.parametrize("side,short", [(14.0, "items"), (12.0, "manifolds and items")])
@pytest.mark.parametrize("coloured", [False, True], ids=["reference", "coloured"])
def test_items_beyond_the_estimate(oracle, side, short, coloured):
    """Bodies dropped into each other: more than three manifolds a body, so the
    first step stops, the arrays grow, and the step is taken again."""
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    n = 800
    ctx = Context(0)
    ctx.set_fused(False)
    g, o = GpuWorld(ctx), oracle.OracleWorld("f32")
    for e in (g, o):
        apply_scene(_heap(n, side, 40), e)
        e.set_schedule(int(coloured))
    for step in range(3):
        print(f"{short}: step {step + 1} of 3", flush=True)
        assert g.process(DT, 1, 2) == o.process(DT, 1, 2) == 0
        if step == 0:
            items = ctx.last_counts()["items"]
            assert items > _room(2 * (n + 1) + 1024), items
            assert (items > _room(4 * (n + 1) + 1024)) == (short != "items"), items
        _same(g, o, step)
    for e in (g, o, ctx):
        e.close()


def test_items_beyond_the_estimate_within_a_call(oracle):
    """The same where the step that stops is not the call's last one."""
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    ctx = Context(0)
    ctx.set_fused(False)
    g, o = GpuWorld(ctx), oracle.OracleWorld("f32")
    for e in (g, o):
        apply_scene(_heap(800, 14.0, 40), e)
    for call in range(2):
        ctx.process_batch_handles([g.handle], DT, 1, 2, 3)
        for _ in range(3):
            assert o.process(DT, 1, 2) == 0
        _same(g, o, call)
    for e in (g, o, ctx):
        e.close()


@pytest.mark.parametrize("iters", [4, 16, 17])
@pytest.mark.parametrize("fit", ["16", "7", "1", "1 without room", "none"])
def test_short_of_memory(oracle, monkeypatch, fit, iters):
    """A device with room for less than the step scratch of 16-iteration programs
    (R2D_SCRATCH_LIMIT: a larger piece is refused)."""
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    n, joints = 600, 1200
    caps = [n + 2, 2 * (n + 2), 1, joints, 4 * (n + 2) + 1024, 8 * (n + 2) + 1024, 4 * (n + 2) + 1024,
            joints + 2 * (n + 2) + 1024]
    grown = [_room(x) for x in caps]
    limit = {"16": rule(1, *grown, 16)[0], "7": rule(1, *grown, 7)[0], "1": rule(1, *grown, 1)[0],
             "1 without room": rule(1, *caps, 1)[0], "none": rule(1, *caps, 1)[0] - 1}[fit]
    monkeypatch.setenv("R2D_SCRATCH_LIMIT", str(limit))
    ctx = Context(0)
    ctx.set_fused(False)
    g, o = GpuWorld(ctx), oracle.OracleWorld("f32")
    for e in (g, o):
        apply_scene(_links(n, joints, 41), e)
    for step in range(2):
        rc = g.process(DT, 2, iters)
        if fit == "none":
            assert rc == 3
            break
        assert rc == 0 and o.process(DT, 2, iters) == 0
        _same(g, o, step)
    for e in (g, o, ctx):
        e.close()


@pytest.mark.parametrize("fit", ["16", "1", "none"])
def test_short_of_memory_one_kernel(oracle, monkeypatch, fit):
    """The same for the one-kernel step's slices (a heap that fits its first slices)."""
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    n, iters = 300, 16
    bodies = n + 1
    slices = [4 * bodies + 65, 32 * bodies + 257, 3 * bodies + 64, 3 * bodies + 65]
    limit = rule(2, *[2 * x for x in slices], 1 if fit != "16" else 16)[0] - (fit == "none")
    monkeypatch.setenv("R2D_SCRATCH_LIMIT", str(limit))
    ctx = Context(0)
    g, o = GpuWorld(ctx), oracle.OracleWorld("f32")
    for e in (g, o):
        apply_scene(_heap(n, 20.0, 42), e)
    for step in range(2):
        rc = g.process(DT, 2, iters)
        if fit == "none":
            assert rc == 3
            break
        assert rc == 0 and o.process(DT, 2, iters) == 0
        _same(g, o, step)
    for e in (g, o, ctx):
        e.close()


def test_admission_follows_the_iterations(gpu_ctx):
    """A budget for two worlds at 4 iterations holds only one at 8."""
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.serve import Server
    for iters, at_once in ((4, 2), (8, 1)):
        ws = [GpuWorld(gpu_ctx) for _ in range(2)]
        for k, w in enumerate(ws):
            apply_scene(_heap(1500, 25.0, 50 + k), w)
        budget = sum(w.footprint() for w in ws)
        sv = Server(gpu_ctx, budget, max_worlds=4, collision_iters=iters)
        try:
            assert (sum(w.footprint() for w in ws) > budget) == (iters == 8)
            for w in ws:
                sv.submit(w, 2)
            assert sv.tick()["running"] == at_once
            sv.drain()
            assert sv.stats()["peak_resident_bytes"] <= budget
        finally:
            sv.close()
            for w in ws:
                w.close()
