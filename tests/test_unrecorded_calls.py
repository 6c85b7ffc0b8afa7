"""Calls that record no gradient go past the autograd Function: only where nothing would look at it."""
import pytest
import torch
from torch.autograd import forward_ad

import linrec_amd
from linrec_amd import ops


def _pair(requires_grad=False):
    g = torch.Generator().manual_seed(3)
    return [f((3, 40, 6), generator=g, dtype=torch.float64).requires_grad_(requires_grad) for f in (torch.randn, torch.rand)]


@pytest.mark.parametrize("dim", [0, 1, 2, -1, -2])
def test_the_same_values_and_strides_as_a_recorded_call(dim):
    want = linrec_amd.linrec(*_pair(True), dim=dim)
    x, c = _pair()
    for got in (linrec_amd.linrec(x, c, dim=dim), torch.no_grad()(linrec_amd.linrec)(*_pair(True), dim=dim),
                torch.inference_mode()(linrec_amd.linrec)(x, c, dim=dim)):
        assert torch.equal(got, want) and got.stride() == want.stride() and not got.requires_grad and got.grad_fn is None
    assert want.requires_grad


def test_forward_mode_and_transforms_are_refused_as_before():
    x, c = _pair()
    with forward_ad.dual_level():
        dual = forward_ad.make_dual(x, torch.ones_like(x))
        assert not ops._nobody_watches(dual, c)
        with pytest.raises(RuntimeError):
            linrec_amd.linrec(dual, c)
    assert ops._nobody_watches(x, c)
    with pytest.raises(RuntimeError):
        torch.func.vmap(linrec_amd.linrec)(x, c)
    with pytest.raises(RuntimeError):
        torch.func.jvp(lambda a: linrec_amd.linrec(a, c), (x,), (torch.ones_like(x),))


def test_a_traced_call_is_not_a_constant():
    x, c = _pair()
    seen = []
    original = ops._nobody_watches
    try:
        ops._nobody_watches = lambda a, b: seen.append(original(a, b)) or seen[-1]
        traced = torch.jit.trace(lambda a, b: linrec_amd.linrec(a, b), (x, c), check_trace=False)
    finally:
        ops._nobody_watches = original
    assert seen and not any(seen)
    assert any("_LinrecFn" in str(n) for n in traced.graph.nodes()), traced.graph
    other, c2 = torch.randn_like(x), torch.rand_like(c)
    assert torch.equal(traced(other, c2), linrec_amd.linrec(other, c2)) and not torch.equal(traced(other, c2), traced(x, c))
