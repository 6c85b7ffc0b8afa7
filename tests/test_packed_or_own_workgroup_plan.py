"""Which dense short rows are packed and which keep a workgroup of their own (planner only, for 256 compute units)."""
import ctypes

import pytest

from linrec_amd import _native as nat

F32, F16, BF16 = 0, 1, 2


@pytest.fixture(autouse=True)
def full_part():
    old = nat.set_compute_units(256)
    yield
    nat.set_compute_units(old)


def packed(dtype, rows, length, is_bwd, reverse=0):
    p = nat.Plan()
    assert nat.lib().linrec_plan(dtype, None, rows, length, length, 1, reverse, int(is_bwd), None, ctypes.byref(p)) == 0
    return "packed" in nat.kernel_table()[p.kernel_id]


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_16_bit_rows_of_whole_slots_that_fill_their_workgroup(dtype):
    """(a workgroup of one row holds 512, 1024, 2048 or 4096 elements)"""
    for is_bwd, least in ((False, 11), (True, 10)):
        for room in (512, 1024, 2048, 4096):
            for sixteenths in range(9, 17):
                for rows in ((1 << 22) // room * 3 // 2, (1 << 24) // room, (1 << 26) // room):
                    length = room * sixteenths // 16
                    if rows * length >= 1 << 22:
                        assert packed(dtype, rows, length, is_bwd) == (sixteenths < least), (is_bwd, rows, length)
    assert not packed(dtype, 1944, 3392, False) and not packed(dtype, 3728, 1792, True)


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_16_bit_backward_of_rows_off_the_slots(dtype):
    for room in (1024, 2048, 4096):
        for rows in ((1 << 24) // room, (1 << 26) // room):
            assert packed(dtype, rows, room * 13 // 16 + 1, True) and packed(dtype, rows, room * 15 // 16 + 1, False), (rows, room)
            assert not packed(dtype, rows, room * 15 // 16 + 1, True), (rows, room)


@pytest.mark.parametrize("is_bwd", [False, True])
def test_single_precision_rows_of_whole_slots(is_bwd):
    for room in (512, 1024, 2048, 4096):
        for rows in ((1 << 23) // room * 3 // 2, (1 << 26) // room):
            if room < 2048:  # (whole rows have to fill four fifths of a workgroup)
                assert packed(F32, rows, room * 11 // 16, is_bwd), (rows, room)
            assert not packed(F32, rows, room * 13 // 16, is_bwd), (rows, room)
        length = room * 10 // 16
        assert not packed(F32, (1 << 22) // length + 1, length, is_bwd), room  # little work
    assert not packed(F32, 4849, 1584, True) and not packed(F32, 22657, 192, False)


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_16_bit_workgroups_of_eight_waves_that_make_about_one_round(dtype):
    """(a compute unit holds four of them, three in the backward)"""
    for rows, length, is_bwd in [(1707, 3436, True), (1908, 3325, True), (1698, 3353, True), (2200, 3524, False), (2430, 3524, False)]:
        assert not packed(dtype, rows, length, is_bwd), (rows, length)
    for rows, length, is_bwd in [(1300, 3436, True), (4000, 3325, True), (1300, 3427, False), (6000, 3427, False)]:
        assert packed(dtype, rows, length, is_bwd), (rows, length)


def test_single_precision_backward_of_short_rows_that_ran_in_reverse():
    """(its scan runs in ascending order, in which the flat kernels are ahead)"""
    for length in (5, 7, 9, 13, 15, 21, 35, 45, 63):
        for elements in (1 << 22, 1 << 23, 1 << 24, 30 << 20):
            rows = elements // length + 1
            flat = length < 16 or elements > 1 << 22
            assert packed(F32, rows, length, True, reverse=1) == (not flat), (rows, length)
            assert packed(F32, rows, length, True, reverse=0) and packed(F32, rows, length, False, reverse=1), (rows, length)
            if length > 8:
                assert packed(BF16, rows, length, True, reverse=1), (rows, length)
    assert packed(F32, (1 << 24) // 101, 101, True, reverse=1)
