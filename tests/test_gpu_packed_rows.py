"""Several whole rows to a workgroup (packed_kernel.hpp), reached through the planner on fewer compute units than there are."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.util import TOL_NORMWISE, check_close

pytestmark = pytest.mark.gpu


@pytest.fixture
def nat():
    from linrec_amd import _native
    yield _native
    _native.set_compute_units(0)


def _f64(t):
    return t.detach().float().cpu().numpy().astype(np.float64)


def _placed(t, start, dtype):
    """`t` as dense rows `start` elements after 16 bytes, and the whole buffer around it."""
    buf = torch.full((t.numel() + 32,), 7.0, dtype=dtype, device="cuda:0")
    view = buf[start:start + t.numel()].view(t.shape)
    view.copy_(t)
    return view, buf


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_rows_of_every_kind_of_length(nat, dtype, reverse):
    """Lengths from a slot to half of the largest tile, around multiples of a wave's 64 and 128 slots; row counts that leave
    the last workgroup one row or a few; bases at several phases; nothing outside the tensor is written."""
    ve = 4 if dtype == torch.float32 else 8
    tol = {torch.float32: TOL_NORMWISE, torch.bfloat16: 1.05 * 2.0 ** -8, torch.float16: 1.05 * 2.0 ** -11}[dtype]  # one rounding
    names, seen = nat.kernel_table(), set()
    lengths = [ve + 1, 2 * ve - 1, 5 * ve + 3, 33 * ve + 1, 40 * ve - 1, 64 * ve - 1, 64 * ve + 1, 75 * ve, 85 * ve - 3, 128 * ve - 1,
               128 * ve + 1, 150 * ve, 256 * ve - 1, 256 * ve + 1, 400 * ve + 1, 500 * ve + 1, 512 * ve - 1]
    if dtype == torch.float32:
        lengths += [512 * ve + 1, 650 * ve + 1, 1024 * ve - 3]
    for cus, elements in ((4, 70000), (1, 140000)):  # (the second: the geometry of large tensors)
        nat.set_compute_units(cus)
        for L in lengths:
            for start in ([0, 1, ve - 1] if L > 64 * ve else [0]):
                rows = elements // L + 1 + (L % 3)
                g = torch.Generator().manual_seed(L * 5 + start)
                x, dy = (torch.randn(rows, L, generator=g).to(dtype) for _ in range(2))
                c = (torch.rand(rows, L, generator=g) * 1.9 - 0.95).to(dtype)
                xd, cd, dyd = (_placed(t, start, dtype)[0] for t in (x, c, dy))
                outs = [_placed(torch.zeros(rows, L), start, dtype) for _ in range(3)]
                what = f"{dtype} {cus} CUs {rows} x {L} start={start} rev={reverse}"
                k = [names[nat.plan(xd, reverse, b)["kernel_id"]] for b in (False, True)]
                print(what, k, flush=True)
                seen.update(n.split("MODE")[0] + n.split("MODE")[1][:4] for n in k if "packed" in n)
                y = nat.fwd(xd, cd, reverse, out=outs[0][0])
                dx, dc = nat.bwd(dyd, cd, y, reverse, out=(outs[1][0], outs[2][0]))
                torch.cuda.synchronize()
                check_close(y, oracle.fwd(_f64(x), _f64(c), reverse), what + " outputs", tol)
                dx_t, dc_t = oracle.bwd(_f64(dy), _f64(c), _f64(y), reverse)
                check_close(dx, dx_t, what + " d_inputs", tol)
                check_close(dc, dc_t, what + " d_coeffs", tol)
                for view, buf in outs:
                    assert (buf[:start] == 7.0).all() and (buf[start + rows * L:] == 7.0).all(), what
    fwd, bwd = ({4, 8}, {4, 8, 16}) if dtype == torch.float32 else ({4, 8}, {4, 8})
    assert {int(s.split("packed_w")[1].split("_")[0]) for s in seen if s.endswith("_FWD")} == fwd, seen
    assert {int(s.split("packed_w")[1].split("_")[0]) for s in seen if s.endswith("_BWD")} == bwd, seen


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("L", [30, 333])
def test_nonfinite_values_stay_in_their_row(nat, L, reverse):
    """A NaN or an infinity, a product of coefficients that overflows, and a coefficient no row uses leave every other row bit
    for bit as it was."""
    nat.set_compute_units(4)
    names = nat.kernel_table()
    rows = 70000 // L
    g = torch.Generator().manual_seed(L)
    x, dy = (torch.randn(rows, L, generator=g).to("cuda:0") for _ in range(2))
    c = torch.rand(rows, L, generator=g).to("cuda:0")
    x2, c2, dy2 = x.clone(), c.clone(), dy.clone()
    first, last = (L - 1, 0) if reverse else (0, L - 1)
    x2[5, 7] = float("nan")
    c2[6, 20] = float("inf")
    x2[20, last] = float("inf")
    c2[9, first] = float("nan")  # never used by the forward
    c2[40] = 1e30                # products overflow within a few elements (what becomes of the row itself is every scan's own)
    dy2[30, 3] = float("nan")
    dy2[31, first] = float("inf")
    for b in (False, True):
        assert "packed" in names[nat.plan(x, reverse, b)["kernel_id"]]
    base, got = nat.fwd(x, c, reverse), nat.fwd(x2, c2, reverse)
    clean = [r for r in range(rows) if r not in (5, 6, 20, 40)]
    assert torch.equal(got[clean], base[clean])
    assert not torch.isfinite(got[5]).all() and not torch.isfinite(got[6]).all() and not torch.isfinite(got[20]).all()
    before = slice(8, None) if reverse else slice(0, 7)
    assert torch.equal(got[5, before], base[5, before])
    bdx, bdc = nat.bwd(dy, c, base, reverse)
    gdx, gdc = nat.bwd(dy2, c2, base, reverse)
    clean = [r for r in range(rows) if r not in (6, 9, 30, 31, 40)]
    assert torch.equal(gdx[clean], bdx[clean]) and torch.equal(gdc[clean], bdc[clean])
    assert not torch.isfinite(gdx[30]).all() and not torch.isfinite(gdx[31]).all()
