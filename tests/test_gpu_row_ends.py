"""Tile kernels whose waves at a row's ends load whole slots and mask them late (tile_kernel.hpp, ENDS)."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.util import TOL_NORMWISE, check_close

pytestmark = pytest.mark.gpu


def _f64(t):
    return t.detach().float().cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_rows_that_start_or_end_inside_a_slot(dtype, reverse):
    """Every geometry of the table that has the form, at lengths where the row's last wave holds one slot, part of its slots or
    none, rows apart by gaps at every phase, a NaN in the gaps that nobody may use or overwrite."""
    from linrec_amd import _native as nat
    ve = 4 if dtype == torch.float32 else 8
    tol = {torch.float32: TOL_NORMWISE, torch.bfloat16: 1.05 * 2.0 ** -8, torch.float16: 1.05 * 2.0 ** -11}[dtype]  # one rounding
    names, seen = nat.kernel_table(), set()
    for slots in (33, 64, 65, 80, 81, 127, 128, 129, 192, 193, 256, 257, 400, 512, 513, 1000, 1025, 2049, 4097):
        for extra, gap, start, rows in [(-1, 0, 0, 5), (0, 1, 0, 6), (1, 2, 1, 5), (2, ve - 1, ve - 1, 7)]:
            L = slots * ve + extra
            if dtype != torch.float32 and slots > 2049:
                continue
            g = torch.Generator().manual_seed(L + gap)

            def placed(t):
                buf = torch.full((rows * (L + gap) + 2 * ve,), float("nan"), dtype=dtype, device="cuda:0")
                view = buf[start:start + rows * (L + gap)].view(rows, L + gap)[:, :L]
                view.copy_(t)
                return view, buf

            x, dy = (torch.randn(rows, L, generator=g).to(dtype) for _ in range(2))
            c = (torch.rand(rows, L, generator=g) * 1.9 - 0.95).to(dtype)
            (xd, _), (cd, _), (dyd, _) = placed(x), placed(c), placed(dy)
            outs = [placed(torch.zeros(rows, L)) for _ in range(3)]
            k = [names[nat.plan(xd, reverse, b)["kernel_id"]] for b in (False, True)]
            what = f"{dtype} {rows} x {L} gap={gap} start={start} rev={reverse}"
            print(what, k, flush=True)
            seen.update(n.split("tile_ends_")[1].split("_MODE")[0] + n.split("MODE")[1][:4] for n in k if "tile_ends" in n)
            y = nat.fwd(xd, cd, reverse, out=outs[0][0])
            dx, dc = nat.bwd(dyd, cd, y, reverse, out=(outs[1][0], outs[2][0]))
            torch.cuda.synchronize()
            check_close(y, oracle.fwd(_f64(x), _f64(c), reverse), what + " outputs", tol)
            dx_t, dc_t = oracle.bwd(_f64(dy), _f64(c), _f64(y), reverse)
            check_close(dx, dx_t, what + " d_inputs", tol)
            check_close(dc, dc_t, what + " d_coeffs", tol)
            for view, buf in outs:
                assert int(torch.isnan(buf).sum()) == buf.numel() - rows * L, what
    assert nat.gave_up_count() == 0
    wanted = {"w1_s1", "w2_s1", "w4_s1", "w4_s2", "w8_s2"} | ({"w1_s2", "w2_s2", "w4_s4"} if dtype == torch.float32 else set())
    for w in wanted:  # (the widest tiles come with more rows than this: the planner splits few long rows)
        assert {f"{w}_v{ve}_FWD", f"{w}_v{ve}_BWD"} <= seen, (w, seen)


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("dtype,rows,L", [(torch.float32, 1030, 4501), (torch.float32, 1030, 8181), (torch.bfloat16, 1030, 9001),
                                          (torch.bfloat16, 4200, 2048), (torch.bfloat16, 16, 4096), (torch.bfloat16, 16, 4088)])
def test_many_rows_in_the_widest_tiles_and_16_bit_rows_of_whole_slots(dtype, rows, L, reverse):
    from linrec_amd import _native as nat
    tol = TOL_NORMWISE if dtype == torch.float32 else 1.05 * 2.0 ** -8
    g = torch.Generator().manual_seed(L)
    x, dy = (torch.randn(rows, L, generator=g).to(dtype) for _ in range(2))
    c = (torch.rand(rows, L, generator=g) * 1.9 - 0.95).to(dtype)
    xd, cd, dyd = (t.to("cuda:0") for t in (x, c, dy))
    assert "tile_ends" in nat.kernel_table()[nat.plan(xd, reverse)["kernel_id"]]
    y = nat.fwd(xd, cd, reverse)
    dx, dc = nat.bwd(dyd, cd, y, reverse)
    torch.cuda.synchronize()
    check_close(y, oracle.fwd(_f64(x), _f64(c), reverse), "outputs", tol)
    dx_t, dc_t = oracle.bwd(_f64(dy), _f64(c), _f64(y), reverse)
    check_close(dx, dx_t, "d_inputs", tol)
    check_close(dc, dc_t, "d_coeffs", tol)


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("dtype,L,gap", [(torch.float32, 8201, 0), (torch.float32, 8195, 2), (torch.float32, 12287, 1), (torch.float32, 16384, 1),
                                         (torch.bfloat16, 16387, 0), (torch.bfloat16, 17000, 0), (torch.bfloat16, 24575, 3)])
def test_one_workgroup_walks_rows_that_end_inside_a_tile(dtype, L, gap, reverse):
    """Rows of one to three whole tiles and a last one of a slot, of part of its slots, or of all but an element."""
    from linrec_amd import _native as nat
    tol = TOL_NORMWISE if dtype == torch.float32 else 1.05 * 2.0 ** -8
    rows = 300
    g = torch.Generator().manual_seed(L)
    x, dy = (torch.randn(rows, L + gap, generator=g).to(dtype)[:, :L] for _ in range(2))
    c = (torch.rand(rows, L + gap, generator=g) * 1.9 - 0.95).to(dtype)[:, :L]
    xd, cd, dyd = (torch.empty(rows, L + gap, dtype=dtype, device="cuda:0")[:, :L].copy_(t) for t in (x, c, dy))
    assert "stream" in nat.kernel_table()[nat.plan(xd, reverse)["kernel_id"]]
    y = nat.fwd(xd, cd, reverse)
    dx, dc = nat.bwd(dyd, cd, y, reverse)
    torch.cuda.synchronize()
    check_close(y, oracle.fwd(_f64(x), _f64(c), reverse), "outputs", tol)
    dx_t, dc_t = oracle.bwd(_f64(dy), _f64(c), _f64(y), reverse)
    check_close(dx, dx_t, "d_inputs", tol)
    check_close(dc, dc_t, "d_coeffs", tol)
