"""Workloads of the linear-recurrence scan, as a program that uses this package calls it.

A case is one call of `linrec_amd.linrec` on tensors that already lie on the GPU, alone (inference) or with
the gradients of its two inputs through autograd (training).  Three layouts occur in earnest:

* "rows": (batch, channels, time) or (channels, time), the scan axis contiguous;
* "transposed": a (channels, time) view of a dense (time, channels) matrix;
* "time_major": (batch, time, channels), scanned with dim=1, as a layer of a sequence model holds it.
"""
import torch

import linrec_amd

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_MAX_ELEMENTS = 1 << 26  # the largest listed case


def _case(layout, batch, channels, time, dtype="f32", coeffs="uniform", reverse=False, grad=True, name=None):
    case = dict(layout=layout, batch=batch, channels=channels, time=time, dtype=dtype, coeffs=coeffs,
                reverse=reverse, grad=grad)
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # one short sequence batch at inference: what counts is the latency of a call
        _case("rows", 1, 64, 4096, grad=False, name="small_forward"),
        # the same in a training step: three tensors of 1 MB, the host's work and the launches
        _case("rows", 1, 64, 4096, name="small_training"),
        # the README's shape, the headline benchmark
        _case("rows", 1, 512, 65536, name="long_rows"),
        # state-space layer, 8 batches of 2048 channels flattened, coefficients near one, run backwards in time
        _case("rows", 1, 16384, 2048, coeffs="sigmoid", reverse=True, name="state_space_rows"),
        # few very long sequences (audio, genomes): parallelism has to come from the scan axis
        _case("rows", 1, 16, 1048576, coeffs="near1", name="very_long_rows"),
        # many short rows whose scan axis is strided: a transposed view, the largest tensor
        _case("transposed", 1, 262144, 256, name="transposed_short"),
        # (256, 100, L) of the accuracy sweep at a length that is no whole number of slots: rows of odd length
        _case("rows", 256, 100, 333, name="odd_short_rows"),
        # long sequences of odd length, more of them than compute units but not a multiple
        _case("rows", 1, 335, 100001, name="odd_long_rows"),
        # the state-space layer in mixed precision
        _case("rows", 8, 2048, 2048, dtype="bf16", coeffs="sigmoid", name="mixed_precision_rows"),
        # a gated recurrent layer on (batch, time, channels) activations in mixed precision
        _case("time_major", 8, 1024, 4096, dtype="bf16", coeffs="sigmoid", name="mixed_precision_time_major"),
        # the same in single precision: more batches of shorter sequences, fewer channels
        _case("time_major", 16, 512, 2048, coeffs="sigmoid", name="time_major"),
        # one prompt through such a layer at inference
        _case("time_major", 1, 2048, 4096, dtype="bf16", coeffs="sigmoid", grad=False, name="prefill_time_major"),
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm; a third of them are powers of two or
    multiples of 64, the rest are left as they fall, odd ones among them."""
    n = int(round(lo * (hi / lo) ** rng.random()))
    kind = rng.randrange(6)
    if kind == 0:
        n = 1 << max(0, n.bit_length() - 1)
    elif kind == 1 and n >= 64:
        n -= n % 64
    return min(max(n, lo), hi)


def draw(rng):
    layout = rng.choice(["rows", "rows", "transposed", "time_major", "time_major"])
    dtype = rng.choice(["f32", "f32", "bf16", "f16"])
    coeffs = rng.choice(["uniform", "sigmoid", "near1"])
    reverse, grad = rng.random() < 0.3, rng.random() < 0.7
    elements = _spread(rng, 1 << 18, _MAX_ELEMENTS)
    if layout == "rows":
        time = _spread(rng, 16, min(1 << 20, elements))
        batch, channels = 1, max(1, elements // time)
    elif layout == "transposed":
        time = _spread(rng, 256, min(1 << 16, elements // 4))
        batch, channels = 1, elements // time
    else:
        channels = _spread(rng, 64, 4096)
        channels -= channels % rng.choice([64, 64, 8, 1])  # a layer's width is mostly a multiple of 64
        batch = _spread(rng, 1, 32)
        time = min(max(256, elements // (channels * batch)), _MAX_ELEMENTS // (channels * batch))
    return _case(layout, batch, channels, time, dtype, coeffs, reverse, grad)


def _shape(case):
    """(shape in memory, number of elements)"""
    b, c, t = case["batch"], case["channels"], case["time"]
    if case["layout"] == "rows":
        return ((b, c, t) if b > 1 else (c, t)), b * c * t
    if case["layout"] == "transposed":
        return (t, c), c * t
    return (b, t, c), b * c * t


def prepare(case, seed):
    shape, _ = _shape(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]

    def normal():
        return torch.randn(shape, generator=gen, device="cuda")

    def on_axis(t):
        t = t.to(dtype)
        return t.t() if case["layout"] == "transposed" else t

    inputs = on_axis(normal())
    if case["coeffs"] == "sigmoid":      # gates of a trained layer: mostly near one
        coeffs = on_axis(torch.sigmoid(normal() + 2.0))
    elif case["coeffs"] == "near1":      # slow decay
        coeffs = on_axis(0.9 + 0.1 * torch.rand(shape, generator=gen, device="cuda"))
    else:
        coeffs = on_axis(torch.rand(shape, generator=gen, device="cuda"))
    state = dict(inputs=inputs, coeffs=coeffs, reverse=case["reverse"], dim=1 if case["layout"] == "time_major" else -1)
    if case["grad"]:
        inputs.requires_grad_()
        coeffs.requires_grad_()
        state["d_outputs"] = on_axis(normal())
    return state


def run(state):
    inputs, coeffs = state["inputs"], state["coeffs"]
    outputs = linrec_amd.linrec(inputs, coeffs, state["reverse"], dim=state["dim"])
    if "d_outputs" not in state:
        return outputs
    d_inputs, d_coeffs = torch.autograd.grad(outputs, (inputs, coeffs), state["d_outputs"])
    return outputs, d_inputs, d_coeffs


def work(case):
    """Forward: inputs, coeffs -> outputs.  Backward, a call of its own that starts when the gradient of the
    outputs has arrived: d_outputs, coeffs, outputs -> d_inputs, d_coeffs."""
    _, n = _shape(case)
    size = 4 if case["dtype"] == "f32" else 2
    return {"bytes": n * size * (8 if case["grad"] else 3), "flops": n * (5 if case["grad"] else 2)}


def tolerance(case):
    """About four times the largest difference seen between the kernels and the sequential recurrence in
    float64 on the same inputs (outputs and gradients, listed and drawn cases): fp32 1.4e-7 in the 2-norm and
    1.6e-6 elementwise (coefficients near one), fp16 2.1e-4 and 4.9e-4, bf16 1.7e-3 and 3.9e-3 (one rounding)."""
    rel, largest = {"f32": (6e-7, 6e-6), "f16": (8e-4, 2e-3), "bf16": (7e-3, 1.6e-2)}[case["dtype"]]
    return {"rel": rel, "max": largest}


def _scan64(inputs, coeffs):
    """The recurrence along the last axis in float64, by doubling: after the step of distance d every position
    holds the map from 2d positions before it."""
    b, a = inputs.clone(), coeffs.clone()
    a[..., 0] = 0.0
    d = 1
    while d < b.shape[-1]:
        step = a[..., d:] * b[..., :-d]
        b[..., d:] += step
        step = a[..., d:] * a[..., :-d]
        a[..., d:] = step
        d *= 2
    return b


def exact(case, seed):
    """Outputs and gradients by the recurrence in float64, from the inputs in their storage type."""
    state = prepare(case, seed)
    scan_axis = state["dim"]

    def rows(t):  # the scan axis last and running forward
        t = t.detach().double().movedim(scan_axis, -1)
        return t.flip(-1) if case["reverse"] else t

    def back(t):
        return (t.flip(-1) if case["reverse"] else t).movedim(-1, scan_axis)

    inputs, coeffs = rows(state["inputs"]), rows(state["coeffs"])
    outputs = _scan64(inputs, coeffs)
    if not case["grad"]:
        return back(outputs)
    # position l of the gradient's recurrence runs backward and takes the coefficient of l + 1
    shifted = torch.cat([coeffs[..., 1:], torch.zeros_like(coeffs[..., :1])], -1)
    d_inputs = _scan64(rows(state["d_outputs"]).flip(-1), shifted.flip(-1)).flip(-1)
    d_coeffs = torch.zeros_like(d_inputs)
    d_coeffs[..., 1:] = d_inputs[..., 1:] * outputs[..., :-1]
    return back(outputs), back(d_inputs), back(d_coeffs)
