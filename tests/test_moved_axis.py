"""A scan axis other than the last, moved inside the autograd function: the same results, strides and gradients as
moving it outside, and saved-tensor hooks see what is saved."""
import pytest
import torch

import linrec_amd


def _case(device, dtype=torch.float64, shape=(3, 70, 5)):
    g = torch.Generator().manual_seed(2)
    return [f(shape, generator=g, dtype=torch.float64).to(dtype).to(device).requires_grad_(r)
            for f, r in ((torch.randn, True), (torch.rand, True), (torch.randn, False))]


def _same_as_outside(device, dtype, shape, dim, reverse):
    x, c, dy = _case(device, dtype, shape)
    y = linrec_amd.linrec(x, c, reverse, dim=dim)
    got = (y, *torch.autograd.grad(y, (x, c), dy))
    y = linrec_amd.linrec(x.transpose(dim, -1), c.transpose(dim, -1), reverse).transpose(dim, -1)
    want = (y, *torch.autograd.grad(y, (x, c), dy))
    for a, b in zip(got, want):
        assert a.stride() == b.stride() and torch.equal(a, b), (dim, a.stride(), b.stride())


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("dim", [0, 1, -2, -3, 2])
def test_same_as_moving_the_axis_outside(dim, reverse):
    _same_as_outside("cpu", torch.float64, (3, 70, 5), dim, reverse)
    x, c, _ = _case("cpu", shape=(3, 6, 4))
    assert torch.autograd.gradcheck(lambda a, b: linrec_amd.linrec(a, b, reverse, dim=dim), (x, c))


@pytest.mark.parametrize("requires_grad", [False, True])
def test_what_is_no_axis_is_refused(requires_grad):
    """A scan axis that is none raises the same error whether or not a gradient is recorded."""
    x, c = (torch.rand(3, 6, 4, requires_grad=requires_grad) for _ in range(2))
    for dim, error in ((None, TypeError), (1.5, TypeError), ("1", (TypeError, RuntimeError)), (3, IndexError), (-4, IndexError)):
        with pytest.raises(error):
            linrec_amd.linrec(x, c, dim=dim)


def test_saved_tensor_hooks_and_in_place_changes():
    x, c, dy = _case("cpu")
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(tuple(t.shape)), t.clone())[1], lambda t: t):
        y = linrec_amd.linrec(x, c, dim=1)
    assert packed == [(3, 70, 5), (3, 70, 5)]
    with torch.no_grad():
        y.zero_()  # (the hooks saved copies)
    dx, dc = torch.autograd.grad(y, (x, c), dy)
    y2 = linrec_amd.linrec(x, c, dim=1)
    for a, b in zip((dx, dc), torch.autograd.grad(y2, (x, c), dy)):
        assert torch.equal(a, b)
    y2 = linrec_amd.linrec(x, c, dim=1)
    with torch.no_grad():
        y2.add_(1.0)  # a saved result that was changed in place is noticed
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y2, (x, c), dy)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_repeated_batches_on_the_device(dtype):
    """Calls on batches of matrices from remembered arguments: new tensors, tensors that start inside a slot, another
    stream, both directions."""
    for dim in (1, 0):
        for rep in range(3):
            for reverse in (False, True):
                _same_as_outside("cuda:0", dtype, (3, 600, 72), dim, reverse)
    side = torch.cuda.Stream()
    x, c, _ = _case("cuda:0", dtype, (3, 601, 72))
    want = linrec_amd.linrec(x[:, 1:], c[:, 1:], dim=1)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = linrec_amd.linrec(x[:, 1:], c[:, 1:], dim=1)
        off = linrec_amd.linrec(x[:, 1:, 1:], c[:, 1:, 1:], dim=1)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    # (off the 16-byte boundary another kernel takes the call: fp32 sums in another order, one rounding on each side)
    tol = 1e-5 if dtype == torch.float32 else 2.0 ** -7
    assert (off.float() - want[:, :, 1:].float()).abs().max() <= tol * want.float().abs().max()
