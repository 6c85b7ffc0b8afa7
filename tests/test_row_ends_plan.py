"""Which launches of one row to a workgroup take the form whose waves at a row's ends mask late (planner only, for 256 compute
units, of which each holds 32 waves)."""
import ctypes

import pytest

from linrec_amd import _native as nat

F32, F16, BF16 = 0, 1, 2


@pytest.fixture(autouse=True)
def full_part():
    old = nat.set_compute_units(256)
    yield
    nat.set_compute_units(old)


def kernel(dtype, rows, length, is_bwd):
    p = nat.Plan()
    assert nat.lib().linrec_plan(dtype, None, rows, length, length + 3, 1, 0, int(is_bwd), None, ctypes.byref(p)) == 0
    return nat.kernel_table()[p.kernel_id], p.waves, p.slots


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("length,waves", [(3001, 4), (6001, 8), (12001, 16)])
def test_backward_of_two_slots_to_a_lane(dtype, length, waves):
    """Its registers leave six or seven waves to a SIMD instead of eight."""
    for eighths in (3, 4, 5, 6, 7, 8, 9, 12, 24, 40):
        rows = -(-eighths * 1024 // waves) + 1
        name, w, s = kernel(dtype, rows, length, True)
        if "tile" in name:
            assert (w, s) == (waves, 2)
            other = 4 <= eighths <= (7 if dtype == BF16 else 5) or (dtype == BF16 and waves == 16 and eighths >= 4)
            assert ("tile_ends" in name) == (not other), (rows, length, eighths, name)


def test_calls_that_were_slower():
    for dtype, rows, length, is_bwd in [(BF16, 2910, 9843, True), (BF16, 2478, 8195, True), (BF16, 559, 7138, True), (BF16, 1206, 4084, True),
                                        (F16, 640, 6001, True), (BF16, 300, 10041, False), (F32, 3065, 549, True)]:
        assert "tile_ends" not in kernel(dtype, rows, length, is_bwd)[0], (dtype, rows, length)
    for dtype, rows, length, is_bwd in [(F16, 2910, 9843, True), (BF16, 2910, 9843, False), (BF16, 100, 9843, True), (BF16, 2000, 7138, True),
                                        (F32, 4500, 549, True)]:
        assert "tile_ends" in kernel(dtype, rows, length, is_bwd)[0], (dtype, rows, length)
