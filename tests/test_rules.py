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
