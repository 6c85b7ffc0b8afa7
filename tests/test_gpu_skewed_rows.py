"""fp32 drift kernels on rows that start or end inside a 16-byte slot (drift_kernel.hpp, SKEWED)."""
import pytest
import torch

from tests.util import check_close, make_inputs, truth

pytestmark = pytest.mark.gpu


def _at_phase(t, start, gap):
    """`t` (rows, length) with `gap` elements between its rows and its base `start` elements after 16 bytes."""
    rows, length = t.shape
    buf = torch.full((rows * (length + gap) + 8,), float("nan"), device="cuda:0")
    view = buf[start:start + rows * (length + gap)].view(rows, length + gap)[:, :length]
    view.copy_(t)
    return view


@pytest.mark.parametrize("reverse", [False, True])
def test_rows_at_every_phase(reverse):
    """Lengths around whole tiles (some rows' last tile then holds no slot at all), every phase of the base, rows apart by
    odd numbers of elements, teams that divide a row's tiles and teams that do not; what lies between rows stays as it was."""
    from linrec_amd import _native as nat
    names = nat.kernel_table()
    forward, backward = [(16, 2, 8192), (8, 4, 8192)], [(16, 1, 4096)]
    for rows, tiles, extra, gap in [(5, 3, -1, 0), (7, 3, 1, 0), (4, 4, -2, 1), (9, 3, 2, 3), (3, 5, 0, 1), (6, 3, -3, 0), (2, 3, 4, 2),
                                    (1, 4, 1, 0), (40, 2, 3, 0)]:
        for start in range(4):
            length = tiles * 8192 + extra
            x, c, dy = make_inputs((rows, length), "near1", seed=length + rows)
            y_t, dx_t, dc_t = truth(x, c, dy, reverse)
            xd, cd, dyd = (_at_phase(t, start, gap) for t in (x, c, dy))
            if start == 0 and (length + gap) % 4 == 0 and length % 4 == 0:
                continue  # (rows of whole slots)
            y = None
            for is_bwd, geometries in ((False, forward), (True, backward)):
                for waves, slots, tile in geometries:
                    count = -(-(length + (0 if start == 0 and (length + gap) % 4 == 0 else 3)) // tile)
                    for team in sorted({1, 2, min(3, count), count}):
                        tuning = nat.Tuning(nat.FAMILY_DRIFT, waves, slots, -1, team)
                        what = f"{rows} x {length} start={start} gap={gap} rev={reverse} waves={waves} slots={slots} team={team}"
                        print(what, "backward" if is_bwd else "forward", flush=True)
                        p = nat.plan(xd, reverse, is_bwd, tuning)
                        assert "drift_skewed" in names[p["kernel_id"]] and (p["tiles_per_row"], p["tasks"]) == (count, team), p
                        out = [_at_phase(torch.zeros(rows, length), start, gap).fill_(7.0) for _ in range(2)]
                        if not is_bwd:
                            y = nat.fwd(xd, cd, reverse, tuning, out=out[0])
                            torch.cuda.synchronize()
                            check_close(y, y_t, what + " outputs")
                        else:
                            nat.bwd(dyd, cd, y, reverse, tuning, out=tuple(out))
                            torch.cuda.synchronize()
                            check_close(out[0], dx_t, what + " d_inputs")
                            check_close(out[1], dc_t, what + " d_coeffs")
                        if gap:
                            between = out[0].as_strided((rows - 1, gap), (length + gap, 1), out[0].storage_offset() + length)
                            assert torch.isnan(between).all(), what
    assert nat.gave_up_count() == 0


@pytest.mark.parametrize("reverse", [False, True])
def test_the_planners_choice_and_a_wait_that_runs_out(reverse):
    """Backward through the default plan at sizes the planner gives to these kernels, then with a poll limit of one."""
    from linrec_amd import _native as nat
    names = nat.kernel_table()
    for rows, length in [(300, 65539), (130, 100001), (20, 700001)]:
        x, c, dy = make_inputs((rows, length), "near1", seed=rows)
        y_t, dx_t, dc_t = truth(x, c, dy, reverse)
        xd, cd, dyd, yd = (t.to("cuda:0") for t in (x, c, dy, torch.from_numpy(y_t).float()))
        p = nat.plan(xd, reverse, True)
        assert "drift_skewed" in names[p["kernel_id"]], p
        for limit in (None, 1):
            old = nat.lib().linrec_set_spin_limit(limit) if limit else None
            try:
                y = nat.fwd(xd, cd, reverse)
                dx, dc = nat.bwd(dyd, cd, yd, reverse)
                torch.cuda.synchronize()
            finally:
                if limit:
                    nat.lib().linrec_set_spin_limit(old)
            check_close(y, y_t, f"{rows} x {length} limit {limit} outputs")
            check_close(dx, dx_t, f"{rows} x {length} limit {limit} d_inputs")
            check_close(dc, dc_t, f"{rows} x {length} limit {limit} d_coeffs")
            if limit is None:
                assert nat.gave_up_count() == 0
        for ws in list(nat._workspaces.values()):
            ws[:16].view(torch.int32)[1] = 0  # (the other tests take a count of zero as the sign that nobody had to fall back)
