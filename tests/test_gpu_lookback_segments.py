"""Segments of a strided scan axis chained by look-back in one launch (collook_kernel.hpp)."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.util import check_close

pytestmark = pytest.mark.gpu

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# max|got - truth| / max|truth|: one rounding of the storage type and 1 % for the fp32 sums before it
# (fp32: the bar of all fp32 kernels)
TOL = {"f32": 1e-5, "f16": 1.01 * 2.0 ** -11, "bf16": 1.01 * 2.0 ** -8}


@pytest.fixture(scope="module")
def nat():
    from linrec_amd import _native
    return _native


def f64(t):
    return t.detach().cpu().double().numpy()


def draw(shape, dtype, seed, near1=False):
    """x, c, dy on the device, (batch, time, channels)"""
    g = torch.Generator().manual_seed(seed)
    x, c, dy = (f(shape, generator=g) for f in (torch.randn, torch.rand, torch.randn))
    if near1:
        c = 1.0 - 0.01 * c
    return [t.to(dtype).to("cuda:0") for t in (x, c, dy)]


def nan_like(t):
    return torch.empty_strided(t.size(), t.stride(), dtype=t.dtype, device=t.device).fill_(float("nan"))


def check_fwd(nat, kind, x, c, reverse, tuning, what):
    y = nat.fwd(x, c, reverse, tuning, out=nan_like(x))
    torch.cuda.synchronize()
    check_close(y, oracle.fwd(f64(x), f64(c), reverse, dtype=np.float64), what + " outputs", TOL[kind])
    return y


def check_bwd(nat, kind, dy, c, y, reverse, tuning, what):
    dx, dc = nat.bwd(dy, c, y, reverse, tuning, out=(nan_like(y), nan_like(y)))
    torch.cuda.synchronize()
    dx_t, dc_t = oracle.bwd(f64(dy), f64(c), f64(y), reverse, dtype=np.float64)
    check_close(dx, dx_t, what + " d_inputs", TOL[kind])
    check_close(dc, dc_t, what + " d_coeffs", TOL[kind])


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("kind", list(DTYPES))
def test_every_geometry_at_its_edges(nat, kind, reverse):
    """Axes around whole segments, rows that leave lanes idle, waves whose lanes belong to different batches."""
    fwd = [(2, 16, 16), (1, 8, 16)] if kind == "f32" else [(4, 16, 16), (2, 16, 16), (1, 8, 16)]
    bwd = [(4, 16, 8), (2, 16, 8), (1, 8, 16)] if kind == "f32" else fwd
    for shape in [(1, 2, 4), (1, 127, 8), (2, 129, 64), (1, 255, 260), (1, 256, 132), (3, 257, 100), (5, 513, 24), (2, 2500, 2),
                  (1, 3000, 66), (7, 1025, 33)]:
        x, c, dy = (t.transpose(1, 2) for t in draw(shape, DTYPES[kind], sum(shape), near1=shape[1] > 1000))
        y = None
        for is_bwd, geometries in ((False, fwd), (True, bwd)):
            for vec, waves, run in geometries:
                if shape[2] % vec:
                    continue
                tuning = nat.Tuning(nat.FAMILY_SEGMENT, vec, run, 1, waves)
                what = f"{kind} {shape} rows/lane={vec} waves={waves} run={run} rev={reverse}"
                print(what, "backward" if is_bwd else "forward", flush=True)
                p = nat.plan(x, reverse, is_bwd, tuning)
                assert (p["family"], p["carry"], p["vec"], p["block"], p["tasks"]) == (nat.FAMILY_SEGMENT, 1, vec, 64 * waves, waves * run), p
                assert p["tiles_per_row"] == -(-shape[1] // (waves * run))
                assert p["grid"] == -(-(shape[0] * shape[2]) // (64 * vec)) * p["tiles_per_row"]
                if is_bwd:
                    check_bwd(nat, kind, dy, c, y, reverse, tuning, what)
                else:
                    y = check_fwd(nat, kind, x, c, reverse, tuning, what)
        assert nat.gave_up_count() == 0


@pytest.mark.parametrize("kind", list(DTYPES))
def test_planner_takes_them_for_batches_whatever_the_strides(nat, kind):
    """The public operator on the forms a batch of matrices comes in: dense, channels cut out of wider ones, views that
    start inside a slot, time outermost, odd channel counts."""
    import linrec_amd
    dtype = DTYPES[kind]
    forms = {
        "dense": ((3, 1100, 200), lambda t: t),
        "wide": ((2, 1100, 300), lambda t: t[:, :, :200]),
        "offset": ((2, 1101, 204), lambda t: t[:, 1:, 3:203]),
        "odd": ((5, 1100, 77), lambda t: t),
        "time outermost": ((1100, 3, 160), lambda t: t[:, :, :128].transpose(0, 1)),
        "two batch dims": ((2, 3, 1100, 40), lambda t: t),
    }
    for name, (shape, form) in forms.items():
        for reverse in (False, True):
            x, c, dy = (form(t) for t in draw(shape, dtype, 5, near1=True))
            plans = [nat.plan(x.transpose(-1, -2), reverse, b) for b in (False, True)]
            assert all((p["family"], p["carry"]) == (nat.FAMILY_SEGMENT, 1) for p in plans), (name, plans)
            x, c = x.detach().requires_grad_(), c.detach().requires_grad_()
            y = linrec_amd.linrec(x, c, reverse, dim=-2)
            dx, dc = torch.autograd.grad(y, (x, c), dy)
            torch.cuda.synchronize()
            rows = [f64(t.transpose(-1, -2)) for t in (x, c, dy, y)]
            check_close(y.transpose(-1, -2), oracle.fwd(rows[0], rows[1], reverse, dtype=np.float64), f"{kind} {name} outputs", TOL[kind])
            dx_t, dc_t = oracle.bwd(rows[2], rows[1], rows[3], reverse, dtype=np.float64)
            check_close(dx.transpose(-1, -2), dx_t, f"{kind} {name} d_inputs", TOL[kind])
            check_close(dc.transpose(-1, -2), dc_t, f"{kind} {name} d_coeffs", TOL[kind])
    assert nat.gave_up_count() == 0


def test_rows_stay_alone_with_their_non_finite_values(nat):
    x, c, dy = (t.transpose(1, 2) for t in draw((2, 2000, 100), torch.float32, 9))
    x[0, 5, 300] = float("nan")
    c[1, 77, 10] = float("inf")
    clean = torch.ones((2, 100), dtype=torch.bool)
    clean[0, 5] = clean[1, 77] = False
    y = nat.fwd(x, c)
    dx, dc = nat.bwd(dy, c, y)
    torch.cuda.synchronize()
    assert nat.plan(x)["carry"] == 1
    for t in (y, dx, dc):
        ok = torch.isfinite(t).all(-1).cpu()
        assert ok[clean].all()
    assert not torch.isfinite(y).all(-1).cpu()[~clean].any()
    # the first position's coefficient takes no part
    c2 = torch.rand_like(x)
    c2[..., 0] = float("nan")
    x2 = torch.randn_like(x)
    assert torch.isfinite(nat.fwd(x2, c2)).all()


@pytest.mark.parametrize("kind", list(DTYPES))
def test_a_wait_that_runs_out_is_answered_from_the_rows(nat, kind, monkeypatch):
    """A poll limit of 1: a segment that does not find what it looks for at once computes it from the row.  In workspaces
    of its own, whose counts of such waits say that it came to that in either pass."""
    assert nat.gave_up_count() == 0
    for name in ("_workspaces", "_ws_pinned", "_ws_retired", "_ws_cleared_in"):
        monkeypatch.setattr(nat, name, type(getattr(nat, name))())
    x, c, dy = (t.transpose(1, 2) for t in draw((3, 4000, 130), DTYPES[kind], 4, near1=True))
    y0 = nat.fwd(x, c)
    torch.cuda.synchronize()
    assert nat.gave_up_count() == 0
    old, before = nat.lib().linrec_set_spin_limit(1), 0
    try:
        for reverse in (False, True):
            check_fwd(nat, kind, x, c, reverse, None, "poll limit 1")
            forward = nat.gave_up_count()
            check_bwd(nat, kind, dy, c, y0, reverse, None, "poll limit 1")
            both = nat.gave_up_count()
            print("waits that ran out so far:", forward, both, flush=True)
            assert before < forward < both
            before = both
        if kind != "f16":  # (whose largest value the growth exceeds)
            x, c = growing_rows(kind)
            assert nat.plan(x)["carry"] == 1
            want = torch.from_numpy(oracle.fwd(f64(x), f64(c), False, dtype=np.float64)[:, :34])
            got = nat.fwd(x, c)[:, :34].cpu().double()
            assert ((got - want).abs() / want.clamp_min(1e-30)).max() <= TOL[kind]
    finally:
        nat.lib().linrec_set_spin_limit(old)
        torch.cuda.synchronize()


def test_graph_replays_match_the_oracle(nat):
    x, c, dy = (t.transpose(1, 2) for t in draw((4, 1500, 96), torch.float32, 1))
    y, dx, dc = nan_like(x), nan_like(x), nan_like(x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        nat.fwd(x, c, out=y)
        nat.bwd(dy, c, y, out=(dx, dc))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        nat.fwd(x, c, out=y)
        nat.bwd(dy, c, y, out=(dx, dc))
    for rep in range(3):
        for dst, src in zip((x, c, dy), draw((4, 1500, 96), torch.float32, 20 + rep)):
            dst.copy_(src.transpose(1, 2))
        for t in (y, dx, dc):
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        check_close(y, oracle.fwd(f64(x), f64(c), False, dtype=np.float64), f"replay {rep} outputs")
        dx_t, dc_t = oracle.bwd(f64(dy), f64(c), f64(y), False, dtype=np.float64)
        check_close(dx, dx_t, f"replay {rep} d_inputs")
        check_close(dc, dc_t, f"replay {rep} d_coeffs")
        nat.fwd(dy, c)  # the program's own eager work between the replays
    assert nat.gave_up_count() == 0


def test_graphs_captured_on_a_cold_stream_clear_their_own_workspace(nat, monkeypatch):
    """Two graphs captured on a stream that has not launched before: the second one is replayed first, on a workspace
    that holds what an earlier graph of a shared memory pool may have left there, and an eager launch comes between."""
    for name in ("_workspaces", "_ws_pinned", "_ws_retired", "_ws_cleared_in"):
        monkeypatch.setattr(nat, name, type(getattr(nat, name))())
    x, c, dy = (t.transpose(1, 2) for t in draw((4, 1500, 96), torch.float32, 1))
    nat.fwd(x, c)  # (the kernels are loaded, the call is remembered)
    nat.bwd(dy, c, x)
    torch.cuda.synchronize()
    side, graphs, ids = torch.cuda.Stream(), [], []
    key = (0, side.cuda_stream)
    for i in range(2):
        y, dx, dc = nan_like(x), nan_like(x), nan_like(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            nat.fwd(x, c, out=y)
            ids.append(nat._capture_id(side.cuda_stream))
            nat.bwd(dy, c, y, out=(dx, dc))
        graphs.append((graph, y, dx, dc, nat._workspaces[key]))
    assert None not in ids and ids[0] != ids[1], ids
    nat._workspaces[key].fill_(0x5a)
    assert nat.gave_up_count() == 0  # (nothing has been launched: what the buffer holds is no count)
    for rep, which in enumerate((1, 1, 0, 1, 0)):
        graph, y, dx, dc, ws = graphs[which]
        for dst, src in zip((x, c, dy), draw((4, 1500, 96), torch.float32, 30 + rep)):
            dst.copy_(src.transpose(1, 2))
        for t in (y, dx, dc):
            t.fill_(float("nan"))
        ws.fill_(0x5a)
        print("replay", rep, "of graph", which, flush=True)
        graph.replay()
        torch.cuda.synchronize()
        check_close(y, oracle.fwd(f64(x), f64(c), False, dtype=np.float64), f"replay {rep} outputs")
        dx_t, dc_t = oracle.bwd(f64(dy), f64(c), f64(y), False, dtype=np.float64)
        check_close(dx, dx_t, f"replay {rep} d_inputs")
        check_close(dc, dc_t, f"replay {rep} d_coeffs")
        if rep:
            with torch.cuda.stream(side):
                eager = nat.fwd(x, c)
            torch.cuda.synchronize()
            assert torch.equal(eager, y) and all(nat._workspaces[key] is not g[4] for g in graphs)


def growing_rows(kind):
    """Inputs and coefficients, (2, 68, 3000), whose running product overflows where the recurrence does not: nothing is
    put in before position 1300 while the coefficients are 2 (batch 0), and values of 2^-60 grow by 2^130 and shrink
    again (batch 1).  The first half of the rows is meant to be read forwards, the second half, its mirror image, backwards.
    All values are positive, so that every result has a relative error of its own."""
    g = torch.Generator().manual_seed(3)
    x, c = 0.5 + torch.rand((2, 68, 3000), generator=g), 0.5 * torch.rand((2, 68, 3000), generator=g)
    x[0, :, :1300] = 0
    c[0, :, :1300] = 2.0
    for pos in (200, 1300, 2400):
        x[1, :, pos - 60:pos + 260] = 0
        c[1, :, pos - 60:pos] = 0.5
        c[1, :, pos:pos + 130] = 2.0
        c[1, :, pos + 130:pos + 260] = 0.5
    for t in (x, c):
        t[:, 34:] = t[:, 34:].flip(-1)
    return [t.to(DTYPES[kind]).transpose(1, 2).contiguous().to("cuda:0").transpose(1, 2) for t in (x, c)]


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("kind", ["f32", "bf16"])
def test_products_of_a_segment_may_overflow_where_the_values_do_not(nat, kind, reverse):
    """A segment publishes the product of its 128 or 256 coefficients before it knows what enters it."""
    x, c = growing_rows(kind)
    rows = [f64(t) for t in (x, c)]
    saved = torch.ones_like(x)
    fwd = [(2, 16, 16), (1, 8, 16)] if kind == "f32" else [(4, 16, 16), (2, 16, 16), (1, 8, 16)]
    bwd = [(4, 16, 8), (2, 16, 8), (1, 8, 16)] if kind == "f32" else fwd
    for is_bwd, geometries in ((False, fwd), (True, bwd)):
        meant = slice(34, 68) if is_bwd != reverse else slice(0, 34)  # (the gradient's scan runs against the forward's)
        want = oracle.bwd(rows[0], rows[1], f64(saved), reverse, dtype=np.float64)[0] if is_bwd else \
            oracle.fwd(rows[0], rows[1], reverse, dtype=np.float64)
        want = torch.from_numpy(want[:, meant])
        assert want.min() >= 0 and 1e19 < want.max() < 1e30
        for vec, waves, run in geometries:
            tuning = nat.Tuning(nat.FAMILY_SEGMENT, vec, run, 1, waves)
            got = nat.bwd(x, c, saved, reverse, tuning)[0] if is_bwd else nat.fwd(x, c, reverse, tuning)
            torch.cuda.synchronize()
            got = got[:, meant].cpu().double()
            error = ((got - want).abs() / want.clamp_min(1e-30)).max().item()
            what = f"{kind} reverse={reverse} {'backward' if is_bwd else 'forward'} rows/lane={vec} waves={waves} run={run}"
            print(what, f"largest relative error {error:.2e}", flush=True)
            # (a value holds about ten inputs, the powers of two are exact: far below the bar of the other tests)
            assert error <= TOL[kind], what
    assert nat.gave_up_count() == 0
