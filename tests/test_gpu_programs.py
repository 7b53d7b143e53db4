"""The solver's program of rows (csrc/r2d_chain.h) where its shape changes: how
many iterations one program covers, one or several waves, planning in LDS or
in global memory, impulses and momenta in LDS or in global memory, in the
one-kernel step and in the separate launches.  Bit for bit against the oracle."""
import numpy as np
import pytest

from helpers import bits_equal, first_diff

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0


def _links(n, joints, seed):
    """n discs in a loose row on the ground, tied by `joints` distance joints
    (repeats, both kinds, ends on one body and static ends among them),
    motors and fixed positions."""
    from resolve2d_amd import scenes
    rng = np.random.default_rng(seed)
    b = scenes._Builder()
    b.gravity(9.81)
    b.static(b.rect(0.0, -0.5, 200.0, 1.0, mu=0.4))
    ids = [b.disc(1.1 * i, 0.5, 0.5, mu=0.4) for i in range(n)]
    ids.append(b.rect(-3.0, 1.0, 1.0, 2.0, mu=0.3))
    b.static(ids[-1])
    for k in range(joints):
        i, j = (int(x) for x in rng.integers(0, len(ids), 2))
        t = int(rng.integers(0, 4))
        d = abs(i - j) * 1.1 + 0.1
        if t == 0:
            b.joint(0, ids[i], ids[j], target=d, pmax=5.0, pmin=-5.0, beta=1.0)
        elif t == 1:
            b.joint(1, ids[i], ids[j], r1=(0.1, 0.0), r2=(0.0, 0.1), target=d, pmax=5.0, pmin=-5.0, beta=1.0)
        elif t == 2:
            b.joint(2, ids[i], tpos=(1.1 * i, 0.6), pmax=2.0, pmin=-2.0, beta=1.0)
        else:
            b.joint(3, ids[i], target=0.3, pmax=2.0, pmin=-2.0, beta=1.0)
    return b.ops


def _heap(n, side, seed):
    """n overlapping boxes and discs in a square: many contact points a body."""
    from resolve2d_amd import scenes
    rng = np.random.default_rng(seed)
    b = scenes._Builder()
    b.gravity(9.81)
    b.static(b.rect(0.0, -0.5, 100.0, 1.0, mu=0.5))
    for i in range(n):
        x, y = rng.uniform(-side / 2, side / 2), rng.uniform(0.4, side)
        if i % 3:
            b.rect(x, y, 0.9, 0.9, mu=0.5, angle=rng.uniform(0.0, 0.4))
        else:
            b.disc(x, y, 0.45, mu=0.5)
    return b.ops


def _swarm(n, seed):
    """n small discs in one cell: n (n - 1) / 2 candidates, of which few collide."""
    from resolve2d_amd import scenes
    rng = np.random.default_rng(seed)
    b = scenes._Builder()
    b.gravity(9.81)
    for x, y in rng.uniform(4.1, 7.9, (n, 2)):
        b.disc(x, y, 0.01, mu=0.5)
    return b.ops


SCENES = {"links": _links, "heap": _heap, "swarm": _swarm}

# scene, sub-steps, iterations, steps, separate launches, LDS limit, warm
CASES = {
    # what one program covers: 1, 3, 5, all 16 of 16, 10 of 20, 1 of 17; none
    **{f"iterations-{k}-{m}": (("links", 12, 9, 1), 2, k, 6, m == "separate", 0, 0.0)
       for k in (0, 1, 3, 5, 16, 17, 20) for m in ("fused", "separate")},
    "no-sub-steps": (("links", 12, 9, 1), 0, 4, 2, True, 0, 0.0),
    "no-iterations-warm-fused": (("heap", 30, 4.0, 2), 2, 0, 4, False, 0, 0.8),
    "no-iterations-warm-separate": (("heap", 30, 4.0, 2), 2, 0, 4, True, 0, 0.8),
    # 1,300 joints on 40 bodies: the plan does not fit the world's LDS
    "plan-global-fused": (("links", 40, 1300, 3), 2, 4, 3, False, 0, 0.0),
    "plan-several-waves": (("links", 40, 1300, 3), 2, 16, 2, True, 0, 0.0),
    # contact points' impulses beside the bodies' LDS
    "impulses-global-fused": (("heap", 220, 5.0, 4), 2, 4, 3, False, 0, 0.0),
    "impulses-global-warm": (("heap", 220, 5.0, 4), 2, 4, 3, False, 0, 0.8),
    "several-waves": (("heap", 900, 14.0, 5), 2, 4, 3, True, 0, 0.0),
    # momenta in global memory, one wave and several
    "momenta-global-one-wave": (("links", 12, 30, 6), 2, 4, 6, True, 1, 0.0),
    "momenta-global-several": (("heap", 900, 14.0, 5), 2, 4, 3, True, 1, 0.0),
    "momenta-global-warm": (("heap", 300, 9.0, 7), 2, 4, 5, True, 1, 0.8),
    # a heap too large for plans and impulses in LDS
    "heap-6000": (("heap", 6000, 30.0, 8), 1, 2, 2, True, 0, 0.0),
    # the coloured order, its counters in LDS and in global memory
    "coloured": (("heap", 900, 14.0, 5), 2, 4, 3, True, 0, 0.0),
    # more candidates than one kernel scans (4.2 M): their collisions' list
    "candidates-4.5-million": (("swarm", 3000, 10), 1, 2, 2, True, 0, 0.0),
    "coloured-9000": (("heap", 9000, 45.0, 9), 1, 2, 2, True, 0, 0.0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_program_matches_oracle(oracle, name):
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    scene, sub, iters, steps, separate, limit, warm = CASES[name]
    ops = SCENES[scene[0]](*scene[1:])
    ctx = Context(0)
    ctx.set_lds_limit(limit)
    ctx.set_fused(not separate)
    g, o = GpuWorld(ctx), oracle.OracleWorld("f32")
    for e in (g, o):
        apply_scene(ops, e)
        if warm:
            e.set_warm_start(warm)
        if name.startswith("coloured"):
            e.set_schedule(1)
    for step in range(steps):
        print(f"{name}: step {step + 1} of {steps}", flush=True)
        assert g.process(DT, sub, iters) == o.process(DT, sub, iters) == 0
        a, b = g.bodies(), o.bodies()
        assert bits_equal(a, b), (step, first_diff(a, b))
        mg, mo = g.manifolds(), o.manifolds()
        assert mg.shape == mo.shape and bits_equal(mg, mo), (step, first_diff(mg, mo))
    g.close()
    o.close()
    ctx.close()


@pytest.mark.parametrize("worlds", [257, 513])
def test_warm_batch_of_several_worlds_a_cu(oracle, worlds):
    """More warm worlds than CUs: the narrow warm kernel, heaps of 1 to 40 bodies."""
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    ctx = Context(0)
    scenes = [_heap(1 + (7 * k) % 40, 2.0 + k % 3, 20 + k) for k in range(worlds)]
    gs = [GpuWorld(ctx) for _ in scenes]
    for ops, g in zip(scenes, gs):
        apply_scene(ops, g)
        g.set_warm_start(0.8)
    for _ in range(2):
        ctx.process_batch_handles([g.handle for g in gs], DT, 2, 4, 3)
    for k in range(0, worlds, 16):
        o = oracle.OracleWorld("f32")
        apply_scene(scenes[k], o)
        o.set_warm_start(0.8)
        for _ in range(6):
            assert o.process(DT, 2, 4) == 0
        a, b = gs[k].bodies(), o.bodies()
        assert bits_equal(a, b), (k, first_diff(a, b))
        o.close()
    for g in gs:
        g.close()
    ctx.close()


@pytest.mark.parametrize("warm", [0.0, 0.8], ids=["cold", "warm"])
def test_coloured_beside_reference_order(oracle, warm):
    """A coloured world whose slots hold more than eight waves' rows, in one
    batch with a world in the reference order (warm started or not)."""
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    ctx = Context(0)
    ctx.set_fused(False)
    scenes = [_heap(3000, 25.0, 30), _heap(200, 7.0, 31)]
    gs, os = [GpuWorld(ctx) for _ in scenes], [oracle.OracleWorld("f32") for _ in scenes]
    for ops, g, o in zip(scenes, gs, os):
        apply_scene(ops, g)
        apply_scene(ops, o)
    for e in (gs[0], os[0]):
        e.set_schedule(1)
    for e in (gs[1], os[1]):
        e.set_warm_start(warm)
    for step in range(3):
        ctx.process_batch_handles([g.handle for g in gs], DT, 2, 4, 1)
        for k, (g, o) in enumerate(zip(gs, os)):
            assert o.process(DT, 2, 4) == 0
            a, b = g.bodies(), o.bodies()
            assert bits_equal(a, b), (step, k, first_diff(a, b))
    for e in gs + os:
        e.close()
    ctx.close()
