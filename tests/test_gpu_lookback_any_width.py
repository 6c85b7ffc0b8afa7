"""Look-back segments whose lanes take several rows at any alignment, and the order their workgroups are dealt out in
(collook_kernel.hpp): rows off 16 bytes, channel counts that leave a batch's last lane overlapping the one before it,
segment counts around the eight that are dealt out at a time."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.test_gpu_lookback_segments import DTYPES, TOL, check_bwd, check_fwd, draw, f64, nat  # noqa: F401  (nat: fixture)
from tests.util import check_close


@pytest.mark.gpu
@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("kind", list(DTYPES))
def test_several_rows_to_a_lane_at_any_alignment(nat, kind, reverse):  # noqa: F811
    fwd = [(4, 16, 8), (2, 16, 16)] if kind == "f32" else [(4, 16, 16), (2, 16, 16)]
    bwd = [(4, 16, 8), (2, 16, 8)] if kind == "f32" else fwd
    for batch, time, channels in [(1, 300, 5), (1, 2049, 257), (1, 2100, 33), (3, 700, 129), (2, 2300, 66), (5, 257, 7), (1, 513, 1023)]:
        for start in (0, 1):  # the bases on 16 bytes, and one element after
            wide = draw((batch, time, channels + start), DTYPES[kind], channels + start, near1=time > 1000)
            x, c, dy = (t[:, :, start:].transpose(1, 2) for t in wide)
            y = None
            for is_bwd, geometries in ((False, fwd), (True, bwd)):
                for vec, waves, run in geometries:
                    tuning = nat.Tuning(nat.FAMILY_SEGMENT, vec, run, 1, waves)
                    what = f"{kind} {(batch, time, channels, start)} rows/lane={vec} run={run} rev={reverse}"
                    print(what, "backward" if is_bwd else "forward", flush=True)
                    p = nat.plan(x, reverse, is_bwd, tuning)
                    assert (p["carry"], p["vec"], p["tiles_per_row"]) == (1, vec, -(-time // (waves * run))), p
                    assert p["grid"] == -(-(batch * -(-channels // vec)) // 64) * p["tiles_per_row"]
                    if is_bwd:
                        check_bwd(nat, kind, dy, c, y, reverse, tuning, what)
                    else:
                        y = check_fwd(nat, kind, x, c, reverse, tuning, what)
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
