"""Operator layer: torch.library custom ops with fake (meta) functions and the autograd rule.

Mirrors linrec/impl/cuda/ops.py:17-39,85-101 of the reference: a forward op
(inputs, coeffs, reverse) -> outputs, a backward op (d_outputs, coeffs, outputs, reverse) ->
(d_inputs, d_coeffs), autograd saving exactly (coeffs, outputs) plus the flag, and None as the
gradient of `reverse`.  Device tensors run the HIP kernels, host tensors the library's host loop;
the op is chosen by the dispatcher from the tensors' device, never by a silent fallback.
"""
from typing import Tuple

import torch
from torch.autograd import forward_ad

from . import _native

__all__ = ["linrec", "linrec_fwd", "linrec_bwd", "linrec_pipe", "linrec_tile", "linrec_ref"]


@torch.library.custom_op("linrec_amd::linrec_fwd", mutates_args=(), device_types=("cuda", "cpu"))
def linrec_fwd(inputs: torch.Tensor, coeffs: torch.Tensor, reverse: bool = False) -> torch.Tensor:
    return _native.fwd(inputs, coeffs, reverse)


@torch.library.custom_op("linrec_amd::linrec_bwd", mutates_args=(), device_types=("cuda", "cpu"))
def linrec_bwd(d_outputs: torch.Tensor, coeffs: torch.Tensor, outputs: torch.Tensor,
               reverse: bool = False) -> Tuple[torch.Tensor, torch.Tensor]:
    return _native.bwd(d_outputs, coeffs, outputs, reverse)


@linrec_fwd.register_fake
def _fake_fwd(inputs, coeffs, reverse=False):
    # same conditions as linrec/impl/cuda/ops.py:23-30, minus the stride restrictions the kernels lifted
    torch._check(inputs.size() == coeffs.size(), lambda: "linrec: inputs and coeffs differ in size")
    torch._check(inputs.device == coeffs.device, lambda: "linrec: inputs and coeffs on different devices")
    torch._check(inputs.dtype == coeffs.dtype, lambda: "linrec: inputs and coeffs differ in dtype")
    return _native.output_like(inputs if _native.kept_layout(inputs) else inputs.contiguous(), fake=True)


@linrec_bwd.register_fake
def _fake_bwd(d_outputs, coeffs, outputs, reverse=False):
    torch._check(d_outputs.size() == coeffs.size() and coeffs.size() == outputs.size(),
                 lambda: "linrec: d_outputs, coeffs and outputs differ in size")
    torch._check(d_outputs.device == coeffs.device and coeffs.device == outputs.device,
                 lambda: "linrec: d_outputs, coeffs and outputs on different devices")
    torch._check(d_outputs.dtype == coeffs.dtype and coeffs.dtype == outputs.dtype,
                 lambda: "linrec: d_outputs, coeffs and outputs differ in dtype")
    like = outputs if _native.kept_layout(outputs) else outputs.contiguous()
    return _native.output_like(like, fake=True), _native.output_like(like, fake=True)


def _setup_context(ctx, inputs, output):
    _, coeffs, reverse = inputs
    ctx.save_for_backward(coeffs, output)  # the inputs themselves are not needed (ops.py:17-21)
    ctx.reverse = reverse


def _backward(ctx, d_outputs):
    coeffs, outputs = ctx.saved_tensors
    d_inputs, d_coeffs = linrec_bwd(d_outputs, coeffs, outputs, ctx.reverse)
    return d_inputs, d_coeffs, None


torch.library.register_autograd("linrec_amd::linrec_fwd", _backward, setup_context=_setup_context)


class _LinrecFn(torch.autograd.Function):
    """The same forward/backward pair as the registered operator, as a plain autograd Function.
    Eager calls go through this class because the Python dispatch of a custom op costs several
    times the kernels' own launch time on small inputs; traced and compiled calls use the operator."""

    # (The scan axis is moved in _native, out of autograd's sight: three views recorded by autograd, and their three
    # counterparts in the backward, took 40 us of host time a step, as long as the kernels of 2^23 elements.)
    @staticmethod
    def forward(ctx, inputs, coeffs, reverse, dim):
        outputs = _native.fwd(inputs, coeffs, reverse, dim=dim)
        ctx.save_for_backward(coeffs, outputs)
        ctx.reverse, ctx.dim = reverse, dim
        return outputs

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, d_outputs):
        coeffs, outputs = ctx.saved_tensors
        d_inputs, d_coeffs = _native.bwd(d_outputs, coeffs, outputs, ctx.reverse, dim=ctx.dim)
        return d_inputs, d_coeffs, None, None


def _nobody_watches(inputs, coeffs):
    """Nothing would look at an autograd Function around this call: no gradient to record, no forward-mode level open, no
    function transform, no tracer."""
    return (not (torch.is_grad_enabled() and (inputs.requires_grad or coeffs.requires_grad))
            and forward_ad._current_level < 0 and not torch._C._are_functorch_transforms_active()
            and torch._C._get_tracing_state() is None)


def linrec(inputs: torch.Tensor, coeffs: torch.Tensor, reverse: bool = False, *, logc: bool = False,
           dim: int = -1) -> torch.Tensor:
    """y[l] = y[l-1] * coeffs[l] + inputs[l] over the last dim (reverse=True: from the far end).

    Same call as the reference's `linrec.linrec` (linrec/__init__.py:5); differentiable in `inputs`
    and `coeffs`.  Under torch.compile / tracing this is the registered operator
    `linrec_amd::linrec_fwd`; in eager mode it is the equivalent autograd Function.

    `logc` and `dim` are the two extra options of the reference's CPU entry point
    (linrec/impl/python/ops.py:8-14,60): coefficients given as logarithms, and a scan axis other than
    the last.  Both are expressed through the same kernels: exp() in front (its derivative comes from
    autograd, so d_coeffs is the gradient with respect to the logarithms), and a transposed view, which
    the strided kernels scan in place.
    """
    if logc:
        coeffs = torch.exp(coeffs)
    last = dim == -1 or dim == inputs.dim() - 1
    plain = (torch.Tensor, torch.nn.Parameter)  # tensor subclasses (fake, functional, ...) take the operator
    if torch.compiler.is_compiling() or type(inputs) not in plain or type(coeffs) not in plain:
        if last:
            return linrec_fwd(inputs, coeffs, reverse)
        return linrec_fwd(inputs.transpose(dim, -1), coeffs.transpose(dim, -1), reverse).transpose(dim, -1)
    dim = -1 if last else dim
    if _nobody_watches(inputs, coeffs):  # (inference: the Function's own bookkeeping is a quarter of a small call)
        return _native.fwd(inputs, coeffs, reverse, dim=dim)
    return _LinrecFn.apply(inputs, coeffs, reverse, dim)


# The reference exports three variants of the same function (ops.py:60,81,101); here one set of
# kernels serves all of them, chosen per shape by the library.
linrec_pipe = linrec_tile = linrec_ref = linrec
