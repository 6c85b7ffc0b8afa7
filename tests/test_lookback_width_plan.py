"""How many rows a lane of the look-back segments takes (planner only, for 256 compute units)."""
import ctypes

import pytest

from linrec_amd import _native as nat

F32, F16, BF16 = 0, 1, 2


@pytest.fixture(autouse=True)
def full_part():
    old = nat.set_compute_units(256)
    yield
    nat.set_compute_units(old)


def rows_of_a_lane(dtype, batch, time, channels, is_bwd):
    """0: not served by look-back segments."""
    p = nat.Plan()
    assert nat.lib().linrec_plan_batched(dtype, None, batch, channels, time, time * channels, 1, channels, 0, int(is_bwd), None,
                                         ctypes.byref(p)) == 0
    return p.vec if p.family == nat.FAMILY_SEGMENT and p.carry == 1 else 0


def rows_of_a_lane_of_one_matrix(dtype, time, channels, is_bwd):
    p = nat.Plan()
    assert nat.lib().linrec_plan(dtype, None, channels, time, 1, channels, 0, int(is_bwd), None, ctypes.byref(p)) == 0
    return p.vec if p.family == nat.FAMILY_SEGMENT and p.carry == 1 else 0


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("is_bwd", [False, True])
def test_lanes_of_narrow_batches_take_rows_that_start_on_an_access(dtype, is_bwd):
    """(of fewer than 64 channels, 80 in 16-bit storage)"""
    least, seen = 64 if dtype == F32 else 80, set()
    for channels in (24, 25, 26, 28, 29, 37, 42, 48, 50, 55, 58, 60, 63, 65, 66, 75, 79, 81, 90, 98, 150, 222):
        for batch, time in ((3, 40000), (6, 50000), (17, 17000), (115, 4000), (320, 750)):
            vec = rows_of_a_lane(dtype, batch, time, channels, is_bwd)
            if channels < least:
                assert vec == 0 or channels % vec == 0, (batch, time, channels, vec)
            elif vec > 1 and channels % vec:
                seen.add(vec)
    assert 4 in seen, seen
    assert rows_of_a_lane(dtype, 2, 262144, 64, is_bwd) == 2  # (positions that start on lines)


def test_a_forward_that_leaves_much_of_the_chip_idle_takes_one_row_to_a_lane():
    """Two rows to a lane from five eighths of the compute units on, in 16-bit storage where one row would make two workgroups
    for each, five for four where the axis is whole segments of 256 positions."""
    for batch, time, channels, want in [(42, 1560, 64, 1), (2, 4100, 512, 1), (2, 12000, 192, 1), (8, 8842, 64, 1), (16, 1560, 192, 2),
                                        (48, 1560, 64, 2), (20, 4100, 64, 2)]:
        assert rows_of_a_lane(F32, batch, time, channels, False) == want, (batch, time, channels)
    for batch, time, channels, want in [(11, 342, 512, 1), (4, 900, 512, 1), (12, 2730, 64, 1), (2, 2000, 512, 1), (7, 1560, 192, 1),
                                        (9, 2048, 192, 2), (7, 2048, 192, 2), (15, 900, 192, 1), (10, 4100, 64, 1), (16, 4100, 64, 2), (5, 1560, 512, 2), (6, 3000, 192, 1), (8, 3000, 192, 2)]:
        for dtype in (F16, BF16):
            assert rows_of_a_lane(dtype, batch, time, channels, False) == want, (batch, time, channels)


def test_a_forward_on_whole_lines_that_makes_hardly_more_than_one_round():
    """(of workgroups, up to 33/32 of the compute units, is not told from one that makes a round)"""
    for batch, time, channels, want in [(4, 13107, 160, 2), (2, 13107, 320, 2), (2, 21845, 192, 2), (5, 22595, 64, 1), (3, 34342, 64, 1),
                                        (2, 17718, 256, 1)]:
        assert rows_of_a_lane(F32, batch, time, channels, False) == want, (batch, time, channels)
    for batch, time, channels, want in [(10, 13130, 64, 2), (14, 9272, 64, 2), (10, 7379, 128, 4), (15, 1040, 512, 4)]:
        assert rows_of_a_lane(BF16, batch, time, channels, False) == want, (batch, time, channels)


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_16_bit_forwards_a_little_beyond_one_round_keep_four_rows(dtype):
    """(of an even number of channels)"""
    for batch, time, channels, want in [(8, 1323, 1584, 4), (29, 1079, 564, 4), (3, 1310, 4268, 4), (48, 3120, 112, 4), (34, 1277, 472, 4),
                                        (8, 1275, 1812, 4), (5, 5584, 675, 2), (4, 38189, 121, 2)]:
        assert rows_of_a_lane(dtype, batch, time, channels, False) == want, (batch, time, channels)


def test_single_precision_pairs_that_fill_one_round():
    """Rows that start on 16 bytes but not on a line: two to a lane where that makes three quarters of a round to a whole one."""
    for batch, time, channels, want in [(24, 1980, 144, 2), (6, 5535, 208, 2), (7, 2883, 328, 2), (2, 3912, 784, 2), (2, 3826, 912, 2),
                                        (34, 2416, 80, 2), (8, 19774, 36, 1), (11, 7742, 104, 1), (4, 5961, 360, 1), (9, 4646, 100, 1)]:
        assert rows_of_a_lane(F32, batch, time, channels, False) == want, (batch, time, channels)


def test_single_precision_pairs_of_few_rows():
    """Up to 1024 rows of an even number of channels, where one row to a lane would take four times the workgroups."""
    for batch, time, channels, want in [(2, 611013, 54, 2), (2, 659408, 42, 2), (2, 390360, 42, 2), (3, 368823, 30, 2), (2, 176680, 126, 2),
                                        (8, 57222, 126, 2), (3, 690000, 24, 2), (2, 256555, 76, 1), (8, 258805, 24, 1), (3, 103563, 27, 1),
                                        (17, 36332, 24, 1)]:
        assert rows_of_a_lane(F32, batch, time, channels, False) == want, (batch, time, channels)


def test_single_precision_backwards_of_64_to_80_channels_take_pairs():
    for batch, time, channels in [(28, 3768, 74), (4, 214903, 66), (55, 1955, 78), (56, 2269, 66), (27, 25043, 66), (7, 17119, 70)]:
        assert rows_of_a_lane(F32, batch, time, channels, True) == 2, (batch, time, channels)
    assert rows_of_a_lane(F32, 28, 3768, 72, True) == 4 and rows_of_a_lane(F32, 28, 3768, 82, True) == 4


@pytest.mark.parametrize("dtype", [F16, BF16])
def test_16_bit_backwards_of_one_matrix_that_drift_teams_serve_in_one_round(dtype):
    for time, channels, want in [(4864, 3772, 0), (4894, 3540, 0), (2048, 3676, 0), (3390, 3812, 4), (8895, 3772, 4), (9131, 4036, 4),
                                 (2368, 7084, 4)]:
        assert rows_of_a_lane_of_one_matrix(dtype, time, channels, True) == want, (time, channels)


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
def test_sixteen_rows_of_one_matrix_over_the_longest_axes(dtype):
    for time, channels, is_bwd, want in [(495094, 16, True, 0), (482545, 16, True, 0), (440210, 12, True, 0), (430000, 9, True, 0),
                                         (415453, 32, True, 1), (400000, 16, True, 1), (400000, 12, True, 1)]:
        assert rows_of_a_lane_of_one_matrix(dtype, time, channels, is_bwd) == want, (time, channels)
    if dtype != F32:
        for time, channels in [(495094, 16), (440210, 12), (429270, 12), (434490, 11)]:
            assert rows_of_a_lane_of_one_matrix(dtype, time, channels, False) == 0, (time, channels)
