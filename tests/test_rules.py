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
