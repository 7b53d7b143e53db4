"""The host's rules for laying out and launching steps (r2d_debug_rule; no GPU)."""
import ctypes

import pytest


def rule(k, *args, n=8):
    from resolve2d_amd import _native as N
    a = (ctypes.c_uint64 * len(args))(*args)
    out = (ctypes.c_uint64 * n)()
    assert N.load().r2d_debug_rule(k, a, out) == 0
    return list(out)


@pytest.mark.parametrize("iters", list(range(1, 70)) + [127, 128, 1009, 65537])
def test_iterations_overlap_in_programs(iters):
    """Any number of iterations runs in programs that overlap at least four."""
    each, rest = rule(0, iters)[:2]
    assert 1 <= each <= 16 and each >= min(iters, 4)
    assert (iters - rest) % each == 0 and rest < each
    assert each + rest <= 16           # what the static scratch holds
    assert iters > 16 or (each, rest) == (iters, 0)


def _room(x):
    return x + x // 2 + 256


@pytest.mark.parametrize("joints", [0, 100000])
@pytest.mark.parametrize("n", [65540, 1 << 20, 40 << 20])
def test_step_scratch_falls_back_to_less_than_before_programs(n, joints):
    """Without programs an item took 176 bytes, room for 9 items a body and 1.5
    a joint was taken, and the arrays grew by half: 3 KB a body.  The shortest
    programs without room to grow take less, so that no world that fitted is
    refused."""
    est = [4 * n + 1024, 8 * n + 1024, 4 * n + 1024, joints + 2 * n + 1024]
    table = 2 * n

    def now(k, room):
        return rule(1, *[room(x) for x in [n, table, 1, joints] + est], k)[0]

    e, r, m = (_room(x) for x in est[:3])
    before = 84 * _room(n) + 12 * _room(table) + 24 * e + 36 * r + 128 * m + 176 * _room(m + _room(joints))
    assert now(1, lambda x: x) < before
    assert now(1, lambda x: x) < now(1, _room) < now(rule(0, 17)[0] + rule(0, 17)[1], _room) < now(16, _room)


@pytest.mark.parametrize("iters", [1, 4, 16, 17])
@pytest.mark.parametrize("sizes", [[8192], [16] * 40, [300, 50, 1024, 700], [1500, 4096, 2000]],
                         ids=["one", "small", "mixed", "large"])
def test_admission_charges_what_is_allocated(sizes, iters):
    """The charges of a batch's worlds cover what the batch's first step
    allocates beyond an empty one's (256 bytes of alignment an array)."""
    each, rest = rule(0, iters)[:2]
    k = each + rest
    joints = [n // 3 for n in sizes]
    charge = sum(rule(3, n, 2 * n, j, iters)[0] for n, j in zip(sizes, joints))
    N, J, W = sum(sizes), sum(joints), len(sizes)

    def step(n, w, j, e, r, m, i):
        return rule(1, *[_room(x) for x in (n, 2 * n, w, j, e, r, m, i)], k)[0]

    separate = step(N, W, J, 4 * N + 1024, 8 * N + 1024, 4 * N + 1024, J + 2 * N + 1024) - step(0, 0, 0, *[1024] * 4)
    assert charge + 60 * 256 >= separate
    if max(sizes) <= 1024:
        slices = rule(2, 2 * sum(4 * n + 65 for n in sizes), 2 * sum(32 * n + 257 for n in sizes),
                      2 * sum(3 * n + 64 for n in sizes), 2 * sum(3 * n + 65 + j for n, j in zip(sizes, joints)), k)[0]
        assert charge + 60 * 256 >= slices + step(N, W, J, 1, 1, 1, 1) - step(0, 0, 0, 1, 1, 1, 1)


@pytest.mark.parametrize("bodies", [50, 200, 300, 501, 1024])
def test_lds_is_divided_among_the_workgroups_there_at_once(bodies):
    """More worlds than a compute unit's registers hold workgroups: LDS is
    divided by those, not by worlds that wait for them; and so that as many are
    there at once (pieces of 1,280 bytes, 1 KB for fixed variables)."""
    pieces = lambda x: -(-(x + 1024) // 1280)
    share = [[rule(4, worlds, groups, bodies, 2 * bodies)[0] for worlds in range(1, 13)] for groups in range(1, 13)]
    least = share[11][11]
    for groups, row in enumerate(share, 1):
        assert row == sorted(row, reverse=True)
        assert set(row[groups:]) <= {row[groups - 1]}        # no less for the worlds that wait
        for worlds, x in enumerate(row, 1):
            assert pieces(x) * min(worlds, groups, 128 // pieces(least)) <= 128
    assert share[0][0] == 159 * 1024


@pytest.mark.parametrize("coloured,warm", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_wide_chains_can_be_switched_off(coloured, warm):
    """r2d_ctx_set_wide_record(0) narrows the chains of batches whose caller
    chose no variant; a variant of 512 threads (0, 13, 14) stays wide."""
    for worlds in (1, 40, 256):
        assert rule(5, 0, worlds, 5000, coloured, warm, 1)[0] >= 512
        assert rule(5, 0, worlds, 5000, coloured, warm, 0)[0] == 256
    assert rule(5, 0, 257, 5000, coloured, warm, 1)[0] == 256
    for variant in range(15):
        wide = rule(5, variant + 1, 40, 5000, coloured, warm, 0)[0]
        assert (wide >= 512) == (variant in (0, 13, 14)), variant


def test_twelve_waves_for_coloured_worlds_that_fill_them():
    for worlds in (1, 24, 256):
        assert [rule(5, 0, worlds, n, 1, 0, 1)[0] for n in (10, 2999, 3000, 9000)] == [512, 512, 768, 768]
        assert [rule(5, 0, worlds, n, c, w, 1)[0] for n in (10, 9000) for c, w in ((0, 0), (0, 1), (1, 1))] == [512] * 6


def test_autotuner_times_each_shape_once():
    from resolve2d_amd import autotune
    fused = [(v, 0, True) for v in autotune.FUSED_VARIANTS]
    phases = [(v, lim, False) for v in autotune.PHASE_VARIANTS for lim in (0, 1024)]
    for worlds in (1, 256, 257, 1024):
        kept = autotune.distinct(fused + phases, worlds)
        assert [c[0] for c in kept if c[2]] == [1, 2, 4, 5, 10, 11, 13, 14]
        # the library's own rule for the chains' threads
        threads = lambda v: min(512, rule(5, v + 1, worlds, 5000, 0, 0, 1)[0])
        want = []
        for v, lim, _ in phases:
            if (threads(v), lim) not in want:
                want.append((threads(v), lim))
        assert [(threads(v), lim) for v, lim, f in kept if not f] == want
        assert autotune.distinct(kept, worlds) == kept


def test_autotuner_keeps_choices_by_call_and_build(monkeypatch, tmp_path):
    from resolve2d_amd import _native, autotune
    shape = (1024, 512, 262144)
    keys = [autotune.cache_key(shape, 4, 4), autotune.cache_key(shape, 4, 16), autotune.cache_key(shape, 2, 4)]
    lib = tmp_path / "lib.so"
    lib.write_bytes(b"another build")
    monkeypatch.setattr(_native, "LIB_PATH", str(lib))
    keys.append(autotune.cache_key(shape, 4, 4))
    assert len(set(keys)) == 4 and all(k.startswith(autotune.shape_key(shape)) for k in keys)


@pytest.mark.parametrize("waves", [4, 12])
def test_more_iterations_do_not_spread_a_small_world(waves):
    """One wave runs a world in the one-kernel step up to 1,536 items, however
    many iterations (fewer iterations: up to more)."""
    for iters in (4, 8, 16, 17, 100):
        assert [rule(6, n, iters, waves)[0] for n in (0, 1, 400, 1536)] == [1] * 4
        assert rule(6, 1600, iters, waves)[0] > 1
    assert rule(6, 3000, 1, waves)[0] == rule(6, 3000, 2, waves)[0] == 1


@pytest.mark.parametrize("iters", list(range(1, 70)) + [127, 1009])
def test_one_sub_step_has_short_programs_for_slow_plans(iters):
    """A divisor of the iterations, at most a quarter of them or two, shorter
    than the other worlds' programs; only in steps of one sub-step."""
    assert rule(7, 0, iters)[0] == rule(7, 2, iters)[0] == rule(7, 4, iters)[0] == 0
    less = rule(7, 1, iters)[0]
    if less == 0:   # theirs are that short
        assert iters != 2 and rule(0, iters)[0] <= max(2, iters // 4)
    else:
        assert iters % less == 0 and less <= max(2, iters // 4) and less < rule(0, iters)[0]
