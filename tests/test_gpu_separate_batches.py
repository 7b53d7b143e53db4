"""The separate launches where a batch is larger than the compute units (narrow
chains and a share of LDS each) and with narrow chains asked for.  Bit for bit
against the oracle."""
import pytest

from helpers import bits_equal, first_diff
from test_gpu_programs import _heap

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0


def _check(oracle, ctx, scenes, warm, coloured, pick, steps=2):
    from resolve2d_amd.engine import GpuWorld, apply_scene
    ctx.set_fused(False)

    def make(k, w):
        apply_scene(scenes[k], w)
        if coloured and k % 5 == 0:   # (a world is one or the other)
            w.set_schedule(1)
        elif warm and k % 3 != 1:
            w.set_warm_start(0.8)
        return w

    gs = [make(k, GpuWorld(ctx)) for k in range(len(scenes))]
    for _ in range(2):
        ctx.process_batch_handles([g.handle for g in gs], DT, 2, 4, steps)
    for k in pick:
        o = make(k, oracle.OracleWorld("f32"))
        for _ in range(2 * steps):
            assert o.process(DT, 2, 4) == 0
        a, b = gs[k].bodies(), o.bodies()
        assert bits_equal(a, b), (k, first_diff(a, b))
        mg, mo = gs[k].manifolds(), o.manifolds()
        assert mg.shape == mo.shape and bits_equal(mg, mo), (k, first_diff(mg, mo))
        o.close()
    for g in gs:
        g.close()


@pytest.mark.parametrize("limit", [0, 1], ids=["lds", "momenta-global"])
@pytest.mark.parametrize("warm,coloured", [(False, False), (True, False), (False, True), (True, True)],
                         ids=["cold", "warm", "coloured", "warm-coloured"])
def test_more_worlds_than_compute_units(oracle, warm, coloured, limit):
    """257 worlds of 1 to 40 bodies, and among them heaps whose plan (20 bytes an
    item), impulses (8 a point) and colours (20 a body) a share of LDS does not
    hold: 24 KB for 600 bodies."""
    from resolve2d_amd.solver import Context
    ctx = Context(0)
    ctx.set_lds_limit(limit)
    dense = {0: (600, 11.0), 57: (600, 12.0), 128: (300, 7.0), 255: (450, 10.0), 256: (200, 5.0)}
    scenes = [_heap(*dense[k], 60 + k) if k in dense else _heap(1 + (7 * k) % 40, 2.0 + k % 3, 60 + k) for k in range(257)]
    _check(oracle, ctx, scenes, warm, coloured, list(dense) + list(range(3, 257, 16)))
    ctx.close()


@pytest.mark.parametrize("warm,coloured", [(False, False), (True, False), (False, True)], ids=["cold", "warm", "coloured"])
def test_narrow_chains(oracle, warm, coloured):
    from resolve2d_amd.solver import Context
    ctx = Context(0)
    ctx.set_wide_record(False)
    scenes = [_heap(900, 14.0, 90), _heap(200, 7.0, 91), _heap(20, 3.0, 92)]
    _check(oracle, ctx, scenes, warm, coloured, range(3))
    ctx.close()
