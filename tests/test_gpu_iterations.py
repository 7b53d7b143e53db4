"""Iteration counts beyond 16 that no program of 4 to 16 iterations divides: the
solver runs programs of four and a shorter one for the rest.  Bit for bit
against the oracle in every form a plan takes, and not slower than the next
count that needs no such program."""
import time

import pytest

from helpers import bits_equal, first_diff
from test_gpu_programs import SCENES

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0

# scene, separate launches, LDS limit, warm, coloured
FORMS = {
    "one-wave": (("links", 12, 9, 1), False, 0, 0.0, False),
    "one-wave-separate": (("links", 12, 9, 1), True, 0, 0.0, False),
    "one-wave-warm": (("heap", 30, 4.0, 2), False, 0, 0.8, False),
    "several-waves": (("heap", 500, 10.0, 5), False, 0, 0.0, False),
    "several-waves-separate": (("heap", 500, 10.0, 5), True, 0, 0.0, False),
    "plan-global": (("links", 40, 1300, 3), False, 0, 0.0, False),
    "plan-global-separate": (("links", 60, 8000, 3), True, 0, 0.0, False),
    "momenta-global-warm": (("heap", 300, 9.0, 7), True, 1, 0.8, False),
    "coloured": (("heap", 500, 10.0, 5), True, 0, 0.0, True),
}


@pytest.mark.parametrize("iters", [17, 19, 34])
@pytest.mark.parametrize("form", list(FORMS))
def test_rest_program_matches_oracle(oracle, form, iters):
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    scene, separate, limit, warm, coloured = FORMS[form]
    ctx = Context(0)
    ctx.set_lds_limit(limit)
    ctx.set_fused(not separate)
    g, o = GpuWorld(ctx), oracle.OracleWorld("f32")
    for e in (g, o):
        apply_scene(SCENES[scene[0]](*scene[1:]), e)
        if warm:
            e.set_warm_start(warm)
        if coloured:
            e.set_schedule(1)
    for step in range(3):
        print(f"{form}, {iters} iterations: step {step + 1} of 3", flush=True)
        assert g.process(DT, 2, iters) == o.process(DT, 2, iters) == 0
        a, b = g.bodies(), o.bodies()
        assert bits_equal(a, b), (step, first_diff(a, b))
        mg, mo = g.manifolds(), o.manifolds()
        assert mg.shape == mo.shape and bits_equal(mg, mo), (step, first_diff(mg, mo))
    for e in (g, o, ctx):
        e.close()


def test_prime_counts_keep_the_overlap():
    """20-row pyramid, 17 and 19 iterations: no longer than five steps of four
    take (one at a time they took nine times a step of four)."""
    from resolve2d_amd import scenes
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    ctx = Context(0)
    w = GpuWorld(ctx)
    apply_scene(scenes.pyramid(rows=20), w)

    def best(iters):
        ts = []
        for _ in range(6):
            t = time.perf_counter()
            ctx.process_batch_handles([w.handle], DT, 4, iters, 4)
            ts.append(time.perf_counter() - t)
        return min(ts[1:])

    ctx.process_batch_handles([w.handle], DT, 4, 4, 10)
    four = best(4)
    for iters in (17, 19):
        assert best(iters) < 5 * four, (iters, best(iters), four)
    w.close()
    ctx.close()


@pytest.mark.parametrize("iters", [2, 3, 5, 8, 10, 16, 31])
@pytest.mark.parametrize("form", ["one-wave", "one-wave-separate", "several-waves-separate", "plan-global-separate",
                                  "momenta-global-warm", "coloured", "large-fused"])
def test_one_sub_step(oracle, form, iters):
    """One sub-step: worlds that are slow to plan run short programs."""
    from resolve2d_amd.engine import GpuWorld, apply_scene
    from resolve2d_amd.solver import Context
    scene, separate, limit, warm, coloured = FORMS.get(form, (("heap", 900, 14.0, 5), False, 0, 0.0, False))
    ctx = Context(0)
    ctx.set_lds_limit(limit)
    ctx.set_fused(not separate)
    g, o = GpuWorld(ctx), oracle.OracleWorld("f32")
    for e in (g, o):
        apply_scene(SCENES[scene[0]](*scene[1:]), e)
        if warm:
            e.set_warm_start(warm)
        if coloured:
            e.set_schedule(1)
    for step in range(3):
        print(f"{form}, {iters} iterations: step {step + 1} of 3", flush=True)
        assert g.process(DT, 1, iters) == o.process(DT, 1, iters) == 0
        a, b = g.bodies(), o.bodies()
        assert bits_equal(a, b), (step, first_diff(a, b))
        mg, mo = g.manifolds(), o.manifolds()
        assert mg.shape == mo.shape and bits_equal(mg, mo), (step, first_diff(mg, mo))
    for e in (g, o, ctx):
        e.close()
