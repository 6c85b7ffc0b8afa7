"""Look-back segments whose lanes take several rows at any alignment, and the order their workgroups are dealt out in
(collook_kernel.hpp): rows off 16 bytes, channel counts that leave a batch's last lane overlapping the one before it,
segment counts around the eight that are dealt out at a time."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.test_gpu_lookback_segments import DTYPES, TOL, check_bwd, check_fwd, draw, f64, nat  # noqa: F401  (nat: fixture)
from tests.util import check_close


@pytest.fixture
def compute_units(nat):  # noqa: F811
    yield nat.set_compute_units
    nat.set_compute_units(0)


@pytest.mark.gpu
@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("kind", list(DTYPES))
def test_several_rows_to_a_lane_at_any_alignment(nat, compute_units, kind, reverse):  # noqa: F811
    """On fewer compute units than there are, so that small tensors get wide accesses: every width, both passes."""
    seen = set()
    for cus, batch, time, channels in [(2, 3, 1100, 129), (3, 2, 2300, 66), (16, 1, 2100, 203), (16, 1, 5000, 131), (8, 1, 1500, 101),
                                       (9, 2, 2100, 257), (16, 2, 3000, 203), (20, 1, 2100, 257), (40, 3, 1100, 205)]:
        compute_units(cus)
        for start in (0, 1):  # the bases on 16 bytes, and one element after
            wide = draw((batch, time, channels + start), DTYPES[kind], channels + start, near1=time > 1000)
            x, c, dy = (t[:, :, start:].transpose(1, 2) for t in wide)
            plans = [nat.plan(x, reverse, b) for b in (False, True)]
            what = f"{kind} {cus} CUs {(batch, time, channels, start)} rows/lane={[p['vec'] for p in plans]} rev={reverse}"
            print(what, flush=True)
            for is_bwd, p in enumerate(plans):
                assert (p["family"], p["carry"]) == (nat.FAMILY_SEGMENT, 1) and p["tiles_per_row"] == -(-time // p["tasks"]), (what, p)
                assert p["grid"] == -(-(batch * -(-channels // p["vec"])) // 64) * p["tiles_per_row"], (what, p)
                seen.add((is_bwd, p["vec"]))
            y = check_fwd(nat, kind, x, c, reverse, None, what)
            check_bwd(nat, kind, dy, c, y, reverse, None, what)
    assert {(0, 4), (0, 2), (1, 4), (1, 2)} <= seen, seen
    assert nat.gave_up_count() == 0


@pytest.mark.gpu
@pytest.mark.parametrize("kind", list(DTYPES))
def test_segments_dealt_out_eight_at_a_time(nat, kind):  # noqa: F811
    """15 to 25 segments of two and of five blocks: none, one, two and three whole groups of eight, and the rest of one."""
    vec, waves, run = 1, 8, 16
    tuning = nat.Tuning(nat.FAMILY_SEGMENT, vec, run, 1, waves)
    for channels in (70, 300, 320):
        for segments in (8, 15, 16, 17, 24, 25):
            time = 128 * segments - 3
            x, c, dy = (t.transpose(1, 2) for t in draw((1, time, channels), DTYPES[kind], segments, near1=True))
            y = check_fwd(nat, kind, x, c, False, tuning, f"{kind} {channels} x {segments} segments")
            check_bwd(nat, kind, dy, c, y, False, tuning, f"{kind} {channels} x {segments} segments")
    assert nat.gave_up_count() == 0


@pytest.mark.gpu
@pytest.mark.parametrize("kind", list(DTYPES))
def test_the_planner_takes_single_matrices_to_them(nat, kind):  # noqa: F811
    """Through the public operator: one matrix whose rows are off 16 bytes, or few, as a transposed view."""
    import linrec_amd
    for time, channels in [(2049, 2809), (5000, 1001), (9000, 50), (300, 32771)]:
        for reverse in (False, True):
            x, c, dy = (t[0].t() for t in draw((1, time, channels), DTYPES[kind], channels, near1=True))
            assert all(nat.plan(x, reverse, b)["carry"] == 1 for b in ((False, True) if channels % 8 else (True,))), (time, channels)
            x, c = x.detach().requires_grad_(), c.detach().requires_grad_()
            y = linrec_amd.linrec(x, c, reverse)
            dx, dc = torch.autograd.grad(y, (x, c), dy)
            torch.cuda.synchronize()
            what = f"{kind} {time} x {channels} rev={reverse}"
            check_close(y, oracle.fwd(f64(x), f64(c), reverse, dtype=np.float64), what + " outputs", TOL[kind])
            dx_t, dc_t = oracle.bwd(f64(dy), f64(c), f64(y), reverse, dtype=np.float64)
            check_close(dx, dx_t, what + " d_inputs", TOL[kind])
            check_close(dc, dc_t, what + " d_coeffs", TOL[kind])
