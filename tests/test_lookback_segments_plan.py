"""What the planner decides about segments of a strided scan axis chained by look-back, for 256 compute units.  No GPU."""
import ctypes

import pytest
import torch

from linrec_amd import _native as nat

S = nat.FAMILY_SEGMENT


@pytest.fixture(autouse=True)
def full_part():
    old = nat.set_compute_units(256)
    yield
    nat.set_compute_units(old)


def plan(dtype, batch, time, channels, is_bwd=False, reverse=False, row_stride=1, batch_stride=None, elem_stride=None, tuning=None):
    """The plan of a dense (batch, time, channels) tensor with the bases on 16 bytes, or of other strides; None if refused."""
    es = elem_stride or channels * row_stride
    p = nat.Plan()
    args = (channels, time, row_stride, es)
    tun = ctypes.byref(tuning) if tuning is not None else None
    if batch > 1:
        rc = nat.lib().linrec_plan_batched(nat.DTYPES[dtype], None, batch, channels, time, batch_stride or time * es, row_stride, es,
                                           int(reverse), int(is_bwd), tun, ctypes.byref(p))
    else:
        rc = nat.lib().linrec_plan(nat.DTYPES[dtype], None, *args, int(reverse), int(is_bwd), tun, ctypes.byref(p))
    if rc == -3:
        return None
    assert rc == 0, rc
    return p.asdict()


def chained(p):
    return p["family"] == S and p["carry"] == 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_a_lane_takes_several_rows_only_where_all_lanes_have_some_next_to_each_other(dtype):
    size = torch.empty(0, dtype=dtype).element_size()
    for batch, time, channels in [(2, 262144, 32), (4, 262144, 16), (2, 65536, 16), (3, 100000, 4), (8, 262144, 16), (2, 262144, 48),
                                  (2, 262144, 64), (2, 262144, 128), (500, 16384, 8), (500, 2000, 8), (7, 67656, 48), (16, 8192, 512)]:
        for is_bwd in (False, True):
            p = plan(dtype, batch, time, channels, is_bwd)
            assert chained(p), (batch, time, channels, p)
            rows = batch * channels
            assert p["vec"] == 1 or (2 * rows > -(-rows // (64 * p["vec"])) * 64 * p["vec"] and channels >= 24), (rows, time, p)
            # workgroups of 64 lanes' rows, and a workspace that does not outgrow the tensors
            assert p["grid"] == -(-batch * channels // (64 * p["vec"])) * p["tiles_per_row"]
            assert p["workspace_bytes"] <= max(1 << 16, batch * time * channels * size), (batch, time, channels, p)
    assert plan(dtype, 16, 8192, 512)["vec"] > 1 and plan(dtype, 2, 262144, 64)["vec"] == 2


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_row_limits_follow_the_rows_a_lane_takes(dtype):
    """One row to a lane up to 16384 rows (16-bit storage: 32767), more of them up to 8192 (16384) where a position's rows
    start on a 128-byte line and up to 65536 where they do not."""
    one, lines = (32767, 16384) if dtype != torch.float32 else (16384, 8192)
    for channels, limit in ((23, one), (77, one), (22, one), (30, 65536), (128, lines), (1024, lines), (100, 65536), (1000, 65536)):
        for batch in (limit // channels, limit // channels + 1):
            p = plan(dtype, batch, 3000, channels, True)
            assert chained(p) == (batch * channels <= limit), (batch, channels, p)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_few_channels_and_few_very_long_rows_stay_with_the_three_launches(dtype):
    half = dtype != torch.float32
    for is_bwd in (False, True):
        for batch, time, channels, want in [(32, 4096, 2, False), (500, 300, 3, False), (13, 131071, 2, False), (13, 131072, 2, True),
                                            (12, 65535, 2, True), (32, 4096, 4, True), (8, 65535, 3, True), (9, 65535, 3, False),
                                            (7, 4095, 4, half), (6, 4095, 4, True), (7, 4096, 4, True), (60, 4095, 7, False), (60, 4095, 6, half),
                                            (60, 300, 8, True),
                                            (2, 524289, 16, False), (2, 524288, 16, True), (2, 524289, 31, False), (2, 524289, 32, True),
                                            (7, 524289, 8, False), (8, 524289, 2, True), (2, 131072, 4, True), (2, 131073, 4, False),
                                            (2, 131073, 5, True)]:
            p = plan(dtype, batch, time, channels, is_bwd)
            assert chained(p) == want and p["family"] == S, (batch, time, channels, is_bwd, p)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_column_blocks_keep_short_backwards_and_launches_a_little_beyond_one_round(dtype):
    half = dtype != torch.float32
    f32 = [(256, 1024, True, False), (352, 832, True, False), (352, 1024, True, True), (448, 768, True, True), (1023, 1024, False, False), (1024, 1024, False, True),
           (1200, 832, False, False), (1700, 960, False, False), (1200, 1024, False, False), (2048, 768, False, True), (1200, 640, False, True), (1800, 1024, False, True), (640, 832, True, False),
           (1200, 832, True, False), (1400, 960, True, False), (1900, 832, True, True), (1536, 768, True, True)]
    f16 = [(256, 1280, True, False), (351, 2048, True, False), (352, 1536, True, True), (1200, 1792, True, False), (1280, 1792, False, False), (1280, 1792, True, False),
           (1280, 2048, True, False), (1200, 2048, True, True), (1400, 1536, True, True), (1400, 2048, False, True), (263, 1368, True, False),
           (264, 1368, True, True)]
    for time, channels, is_bwd, want in f16 if half else f32:
        p = plan(dtype, 8, time, channels, is_bwd)
        assert chained(p) == want, (time, channels, is_bwd, p)
        assert want or (p["family"], p["carry"]) == (nat.FAMILY_COLUMN, 2), (time, channels, is_bwd, p)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_column_drift_teams_keep_backwards_that_would_take_narrow_accesses(dtype):
    f32 = [(8, 4096, 175, False), (2, 8192, 701, False), (3, 4096, 467, False), (3, 4096, 1365, True), (56, 3132, 47, True),
           (2, 8192, 700, True), (16, 2048, 512, True)]
    f16 = [(2, 3000, 1750, False), (8, 2100, 504, False), (8, 2048, 512, True), (8, 4096, 1024, True), (3, 4096, 1344, True)]
    for batch, time, channels, want in f32 if dtype == torch.float32 else f16:
        p = plan(dtype, batch, time, channels, True)
        assert chained(p) == want and (want or p["family"] == nat.FAMILY_COLDRIFT), (batch, time, channels, p)
        assert chained(plan(dtype, batch, max(time, 4096), channels))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("channels", [2, 32, 48, 64, 100, 1024])
def test_a_lane_is_less_than_2_31_bytes_from_its_wave(dtype, channels):
    """The kernel adds 32 bits of bytes per lane to an address per wave: the largest batch stride that is accepted keeps
    all rows of a block within them, the next one is refused and planned otherwise."""
    size, time = torch.empty(0, dtype=dtype).element_size(), 4096
    for vec, waves, run in ((1, 8, 16), (2, 16, 16), (4, 16, 16)):
        tuning = nat.Tuning(S, vec, run, 1, waves)
        if plan(dtype, 64, time, channels, tuning=tuning) is None:
            assert (dtype == torch.float32 and vec == 4) or channels % vec  # (no such kernel; rows of a lane in two batches)
            continue
        low, high = time * channels // vec, 1 << 40  # in steps of the rows of a lane, which have to lie in one slot
        while high - low > 1:
            mid = (low + high) // 2
            accepted = plan(dtype, 64, time, channels, batch_stride=mid * vec, tuning=tuning) is not None
            low, high = (mid, high) if accepted else (low, mid)
        rows, worst = 64 * vec, 0
        offset = lambda r: (r // channels) * low * vec + r % channels
        for block in range(64 * channels // rows + 1):
            first, last = block * rows, min(block * rows + rows, 64 * channels) - vec
            if first <= last:
                worst = max(worst, (offset(last) - offset(first) + vec) * size)
        assert worst < 1 << 31, (vec, low, worst)
        assert channels >= rows or worst > 1 << 28, (vec, low, worst)  # (and the bound is no more than a few times too small)
    wide = plan(dtype, 64, time, channels, batch_stride=(1 << 40) + 64)
    assert wide is not None and not chained(wide)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("is_bwd", [False, True])
def test_the_same_where_lanes_share_rows(dtype, is_bwd):
    """Channels that are no multiple of the rows of a lane, which the planner alone takes: a batch's last lane starts early.
    The first batch stride beyond the bound is served otherwise."""
    size, time, seen = torch.empty(0, dtype=dtype).element_size(), 4096, set()
    for batch, channels in ((8, 1025), (8, 1026), (8, 2809), (8, 222), (40, 83), (64, 101)):
        def wide(stride):
            p = plan(dtype, batch, time, channels, is_bwd, batch_stride=stride)
            return p["vec"] if p is not None and chained(p) and channels % p["vec"] else 0
        low = time * channels
        if not wide(low):
            continue
        vec, high = wide(low), 1 << 40
        while high - low > 1:  # (the stride alone does not change the rows of a lane but where one is refused)
            mid = (low + high) // 2
            low, high = (mid, high) if wide(mid) == vec else (low, mid)
        lanes = -(-channels // vec)
        offset = lambda lane: lane // lanes * low + min(lane % lanes * vec, channels - vec)
        blocks = range(0, batch * lanes, 64)
        worst = max((offset(min(b + 64, batch * lanes) - 1) - offset(b) + vec) * size for b in blocks)
        assert worst < 1 << 31, (batch, channels, vec, low, worst)
        assert lanes >= 64 or worst > 1 << 28, (batch, channels, vec, low, worst)
        seen.add(vec)
    assert 4 in seen, seen


def test_strides_that_run_backwards_or_batches_that_overlap_are_refused():
    tuning = nat.Tuning(S, 1, 16, 1, 8)
    assert plan(torch.float32, 4, 4096, 64, tuning=tuning) is not None
    assert plan(torch.float32, 4, 4096, 64, row_stride=-1, elem_stride=64, tuning=tuning) is None
    assert plan(torch.float32, 4, 4096, 64, batch_stride=32, elem_stride=64, tuning=tuning) is None
