"""What a plan costs a call: every call plans anew, so the rules may compare geometries but plan only the one they take."""
import ctypes
import time

import pytest

from linrec_amd import _native as nat


def _fastest(fn, args, calls=500, repeats=40):
    best = float("inf")
    for _ in range(repeats):
        t = time.perf_counter()
        for _ in range(calls):
            fn(*args)
        best = min(best, time.perf_counter() - t)
    return best / calls


@pytest.mark.parametrize("dtype", [0, 2])
@pytest.mark.parametrize("is_bwd", [0, 1])
def test_look_back_segments_are_planned_once(dtype, is_bwd):
    """Well below the cost of a launch of drift teams over 16 x 2^20 floats forward, whose rules go through every size of a
    team (both through the same binding; three geometries planned in full cost more than that, bf16 1.9 to 2.4 us against 1.6)."""
    L, p = nat.lib(), nat.Plan()
    ref = ctypes.byref(p)
    old = nat.set_compute_units(256)
    try:
        teams = _fastest(L.linrec_plan, (0, None, 16, 1 << 20, 1 << 20, 1, 0, 0, None, ref))
        assert p.family == nat.FAMILY_DRIFT
        for batch, time_, channels in [(8, 4096, 1024), (2, 2048, 1024), (16, 2048, 512)]:
            args = (dtype, None, batch, channels, time_, time_ * channels, 1, channels, 0, is_bwd, None, ref)
            cost = _fastest(L.linrec_plan_batched, args)
            if p.family == nat.FAMILY_SEGMENT:
                assert cost < 0.75 * teams, (batch, time_, channels, cost * 1e6, teams * 1e6)
        assert p.family == nat.FAMILY_SEGMENT and p.carry == 1
    finally:
        nat.set_compute_units(old)
