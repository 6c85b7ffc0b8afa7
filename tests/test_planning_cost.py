"""What a plan costs a call: every call plans anew, so the rules may compare geometries but plan only the one they take."""
import ctypes
import time

import pytest

from linrec_amd import _native as nat


def _fastest(*calls, times=300, rounds=60):
    """The smallest time of each of `calls` ((function, arguments)), measured in turn so that a busy host slows all alike."""
    best = [float("inf")] * len(calls)
    for _ in range(rounds):
        for i, (fn, args) in enumerate(calls):
            t = time.perf_counter()
            for _ in range(times):
                fn(*args)
            best[i] = min(best[i], time.perf_counter() - t)
    return [b / times for b in best]


@pytest.mark.parametrize("dtype", [0, 2])
@pytest.mark.parametrize("is_bwd", [0, 1])
def test_look_back_segments_are_planned_once(dtype, is_bwd):
    """Well below the cost of a launch of drift teams over 16 x 2^20 floats forward, whose rules go through every size of a
    team (both through the same binding; three geometries planned in full cost more than that, bf16 1.9 to 2.4 us against 1.6)."""
    L, p, q = nat.lib(), nat.Plan(), nat.Plan()
    old = nat.set_compute_units(256)
    try:
        teams = (L.linrec_plan, (0, None, 16, 1 << 20, 1 << 20, 1, 0, 0, None, ctypes.byref(p)))
        for batch, time_, channels in [(8, 4096, 1024), (2, 2048, 1024), (16, 2048, 512)]:
            segments = (L.linrec_plan_batched, (dtype, None, batch, channels, time_, time_ * channels, 1, channels, 0, is_bwd, None,
                                                ctypes.byref(q)))
            for _ in range(4):
                cost_teams, cost = _fastest(teams, segments)
                if cost < 0.75 * cost_teams:
                    break
            assert p.family == nat.FAMILY_DRIFT and q.family == nat.FAMILY_SEGMENT and q.carry == 1
            assert cost < 0.75 * cost_teams, (batch, time_, channels, cost * 1e6, cost_teams * 1e6)
    finally:
        nat.set_compute_units(old)
