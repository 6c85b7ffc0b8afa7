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


@pytest.fixture
def nat():
    from linrec_amd import _native
    yield _native
    _native.set_compute_units(0)


@pytest.mark.parametrize("reverse", [False, True])
def test_rows_at_every_phase(nat, reverse):
    """Lengths around whole tiles (some rows' last tile then holds no slot at all), every phase of the base, rows apart by
    odd numbers of elements, on fewer compute units than there are, so that small tensors get to these kernels, in teams
    that divide a row's tiles and teams that do not; what lies between rows stays as it was."""
    names = nat.kernel_table()
    teams = set()
    #    CUs, rows, tiles of 8192, and
    for cus, rows, tiles, extra, gap in [(4, 5, 5, -1, 0), (5, 7, 5, 1, 0), (6, 4, 7, -2, 1), (7, 9, 5, 2, 3), (24, 21, 5, 3, 0),
                                         (40, 23, 9, 1, 0), (40, 30, 8, -1, 3)]:
        for start in range(4):
            length = tiles * 8192 + extra
            if start == 0 and (length + gap) % 4 == 0 and length % 4 == 0:
                continue  # (rows of whole slots)
            nat.set_compute_units(cus)
            x, c, dy = make_inputs((rows, length), "near1", seed=length + rows)
            y_t, dx_t, dc_t = truth(x, c, dy, reverse)
            xd, cd, dyd = (_at_phase(t, start, gap) for t in (x, c, dy))
            out = [_at_phase(torch.zeros(rows, length), start, gap).fill_(7.0) for _ in range(3)]
            plans = [nat.plan(xd, reverse, b) for b in (False, True)]
            what = f"{cus} CUs {rows} x {length} start={start} gap={gap} rev={reverse}"
            print(what, [(names[p["kernel_id"]], p["tasks"], p["grid"]) for p in plans], flush=True)
            whole = start == 0 and (gap + length) % 4 == 0
            for p, tile, skewed in ((plans[0], 8192, rows >= 20), (plans[1], 4096, True)):
                if skewed:
                    assert "drift_skewed" in names[p["kernel_id"]] and p["grid"] <= cus, (what, p)
                    assert p["tiles_per_row"] == -(-((length + (0 if whole else 3) + 3) // 4 * 4) // tile), (what, p)
                    teams.add((p["tiles_per_row"] % p["tasks"] == 0, p["tasks"] > 1))
            y = nat.fwd(xd, cd, reverse, out=out[0])
            nat.bwd(dyd, cd, y, reverse, out=tuple(out[1:]))
            torch.cuda.synchronize()
            for got, want, name in ((y, y_t, "outputs"), (out[1], dx_t, "d_inputs"), (out[2], dc_t, "d_coeffs")):
                check_close(got, want, f"{what} {name}")
                if gap:
                    between = got.as_strided((rows - 1, gap), (length + gap, 1), got.storage_offset() + length)
                    assert torch.isnan(between).all(), what
    assert {(True, True), (False, True)} <= teams
    assert nat.gave_up_count() == 0


@pytest.mark.parametrize("reverse", [False, True])
def test_one_row_in_a_team_of_more_than_64(nat, reverse):
    names = nat.kernel_table()
    nat.set_compute_units(128)
    x, c, dy = make_inputs((1, 12 * 8192 * 128 + 5), "near1", seed=2)
    y_t, dx_t, dc_t = truth(x, c, dy, reverse)
    xd, cd, dyd = (t.to("cuda:0") for t in (x, c, dy))
    plans = [nat.plan(xd, reverse, b) for b in (False, True)]
    assert [names[p["kernel_id"]].rsplit("_", 3)[0] for p in plans] == ["drift_skewed_w8_s4", "drift_skewed_w16_s1"], plans
    assert all(p["tasks"] > 64 for p in plans), plans
    y = nat.fwd(xd, cd, reverse)
    dx, dc = nat.bwd(dyd, cd, y, reverse)
    torch.cuda.synchronize()
    for got, want, name in ((y, y_t, "outputs"), (dx, dx_t, "d_inputs"), (dc, dc_t, "d_coeffs")):
        check_close(got, want, name)
    assert nat.gave_up_count() == 0


def test_a_caller_who_names_the_family_gets_rows_of_whole_slots(nat):
    for shape in ((30, 65537), (30, 65538)):
        for is_bwd in (False, True):
            with pytest.raises(NotImplementedError):
                nat.plan(torch.empty(shape), False, is_bwd, nat.Tuning(nat.FAMILY_DRIFT))


@pytest.mark.parametrize("reverse", [False, True])
def test_the_planners_choice_and_a_wait_that_runs_out(nat, reverse):
    """Backward through the default plan at sizes the planner gives to these kernels, then with a poll limit of one."""
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
