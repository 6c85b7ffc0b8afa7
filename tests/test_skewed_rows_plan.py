"""What the planner decides about long fp32 rows that start or end inside a slot, where a row takes one tile more than its
length has (planner only, for 256 compute units)."""
import ctypes

import pytest

from linrec_amd import _native as nat

TILE = 8192  # elements of a tile of the drift kernels' forward


@pytest.fixture(autouse=True)
def full_part():
    old = nat.set_compute_units(256)
    yield
    nat.set_compute_units(old)


def noalloc(rows, length, base=None):
    """(return code, kernel, plan) of a forward that has the library's static scratch array and nothing else."""
    p = nat.Plan()
    rc = nat.lib().linrec_plan_noalloc(nat.DTYPES[nat.torch.float32], base, rows, length, length, 1, 0, None, ctypes.byref(p))
    return rc, nat.kernel_table()[p.kernel_id] if rc == 0 else None, p


def most_tiles():
    """Tiles the static scratch array has descriptors for."""
    low, high = 1, 1 << 20
    while high - low > 1:
        mid = (low + high) // 2
        low, high = (mid, high) if nat.lib().linrec_workspace_bytes_for_tiles(mid) <= 4 << 20 else (low, mid)
    return low


@pytest.mark.parametrize("rows", [1, 2, 3, 5, 7, 200])
def test_a_row_s_last_slot_counts_in_the_workspace(rows):
    """As many tiles as the scratch array holds, by their length: rows at any phase may take one more, and go where rows
    a little longer go."""
    full = most_tiles() // rows * TILE
    for base in (None, 4):
        rc, longer, _ = noalloc(rows, full + 5, base)
        assert rc == 0 and "tile" in longer
        for length in (full - 2, full - 1, full):
            rc, name, p = noalloc(rows, length, base)
            assert rc == 0 and p.workspace_bytes <= 4 << 20 and "stream" not in name, (rows, length - full, base, rc, name)
        rc, name, p = noalloc(rows, full - TILE - 1, base)
        assert rc == 0 and ("drift_skewed" in name or rows * full < 12 * TILE * 256), name


def test_rows_of_as_many_tiles_take_the_same_launch():
    """Rows of whole tiles that start inside a slot take as many tiles as rows an element longer: same teams, same waves."""
    seen = set()
    for rows in (1, 2, 3, 24, 50, 100, 192, 255):
        for tiles in (8, 20, 33, 64, 65, 97, 130, 257, 400, 1025):
            plans = []
            for length in (tiles * TILE, tiles * TILE + 1):
                p = nat.Plan()
                assert nat.lib().linrec_plan(0, 4, rows, length, length, 1, 0, 0, None, ctypes.byref(p)) == 0
                plans.append(p.asdict())
            a, b = plans
            if a["family"] == b["family"] == nat.FAMILY_DRIFT:
                keys = ("waves", "slots", "tiles_per_row", "tasks", "grid", "kernel_id")
                assert [a[k] for k in keys] == [b[k] for k in keys], (rows, tiles, a, b)
                seen.add((a["waves"], a["tasks"] > 64))
    assert {(16, False), (8, True)} <= seen, seen


def test_a_tile_more_does_not_send_rows_elsewhere():
    """Whether drift teams serve rows at any phase is decided by the length alone; their teams may be smaller than four where
    the last slot's tile leaves them nothing better."""
    for cus, rows, length, stride in [(6, 4, 57342, 57343), (6, 4, 57341, 57343), (256, 171, 57342, 57343), (256, 300, 65541, 65541)]:
        nat.set_compute_units(cus)
        p = nat.Plan()
        assert nat.lib().linrec_plan(0, None, rows, length, stride, 1, 0, 1, None, ctypes.byref(p)) == 0
        assert "drift_skewed" in nat.kernel_table()[p.kernel_id], (cus, rows, length)
