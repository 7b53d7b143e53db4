"""A large world's chain in the separate launches by where its state is: the
momenta of the bodies its items touch in LDS and the impulses of its points in
global memory, or both in global memory.  A dense pile of 7,000 bodies, nearly
all touched from the first step, bit for bit against the oracle."""
import pytest

from helpers import bits_equal, first_diff
from resolve2d_amd import scenes
from resolve2d_amd.engine import GpuWorld, apply_scene
from test_gpu_big_chain import _touched

pytestmark = pytest.mark.gpu

# LDS words of a chain alone on its CU; a touched body's momentum takes 4 (and
# 64 spare places), a point's impulses 2 (and a spare one)
WORDS = 159 * 1024 // 4


@pytest.mark.parametrize("limit", [0, 64], ids=["momenta-lds", "momenta-global"])
@pytest.mark.parametrize("warm,coloured", [(0.0, 0), (0.8, 0), (0.0, 1)], ids=["cold", "warm", "coloured"])
def test_impulses_in_global_memory(oracle, warm, coloured, limit):
    from resolve2d_amd.solver import Context
    ctx = Context(0)
    ctx.set_lds_limit(limit)
    ops = scenes.mixed(7000, seed=5, width=60.0, height=60.0, ground_w=80.0)
    g, o = GpuWorld(ctx), oracle.OracleWorld("f32")
    for e in (g, o):
        apply_scene(ops, e)
        if warm:
            e.set_warm_start(warm)
        e.set_schedule(coloured)
    for step in range(6):
        print(f"step {step + 1} of 6", flush=True)
        assert g.process(scenes.DT, 4, 4) == o.process(scenes.DT, 4, 4) == 0
        a, b = g.bodies(), o.bodies()
        assert bits_equal(a, b), (step, first_diff(a, b))
        mg, mo = g.manifolds(), o.manifolds()
        assert mg.shape == mo.shape and bits_equal(mg, mo), (step, first_diff(mg, mo))
        points = len(mo) + int(((mo[:, 7] > 0) & (mo[:, 20] > 0)).sum())
        momenta = 4 * (_touched(o, ops) + 64)
        assert momenta <= WORDS < momenta + 2 * (points + 1), (momenta, points)
    for e in (g, o, ctx):
        e.close()
