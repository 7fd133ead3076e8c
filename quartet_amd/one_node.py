"""The native layer calls as one autograd node of Python, for callers that record or transform what Python runs.

The layers' autograd functions are native (csrc/host_ext.cpp): what they allocate goes through PyTorch's operators, what
they launch does not.  ``torch.jit.trace`` would therefore record the allocations and leave the launches out, and a replay
would return memory nobody wrote.  Under a trace a call goes through a Python autograd function instead, which the
trace keeps as one node that runs the whole call again: packed weights are looked up, and random numbers drawn, on every
replay.  The same function answers where a call has no meaning: it has no forward-mode derivative, so a dual tensor raises
NotImplementedError whether or not anything asks for a gradient (the native call would hand back a tensor without its
tangent), and no rule for ``torch.func``'s transforms, which raise RuntimeError."""
import functools

import torch
from torch.autograd import forward_ad


def transformed():
    """Whether calls are being recorded by a trace, may carry forward-mode tangents or run inside a ``torch.func`` transform.
    Replaced by the native extension's own when that is loaded (the same answer, in a tenth of the time)."""
    return torch.jit.is_tracing() or forward_ad._current_level >= 0 or torch._C._are_functorch_transforms_active()


def use(native):
    global transformed
    transformed = native


class _Unrecorded:
    """What a trace's node runs is the node's own: nothing of it is recorded (and sizes are plain numbers there)."""

    def __enter__(self):
        self.state = torch._C._get_tracing_state()
        torch._C._set_tracing_state(None)

    def __exit__(self, *exc):
        torch._C._set_tracing_state(self.state)


def _seen(t):
    """`t` as a tensor that the trace has seen allocated: one it has not seen would be kept in the recorded graph as a constant."""
    if not (isinstance(t, torch.Tensor) and torch.jit.is_tracing()):
        return t
    seen = torch.empty(0, dtype=t.dtype, device=t.device)
    with _Unrecorded():
        seen.data = t
    return seen


class OneNode(torch.autograd.Function):
    """fn(*args) with the native graph behind its outputs kept inside the node."""

    @staticmethod
    def forward(ctx, fn, *args):
        ctx.set_materialize_grads(False)
        ctx.wanted = ctx.needs_input_grad[1:]
        with _Unrecorded():
            if any(ctx.wanted):
                args = [a.detach().requires_grad_(want) if isinstance(a, torch.Tensor) else a for a, want in zip(args, ctx.wanted)]
                ctx.inner = [a for a, want in zip(args, ctx.wanted) if want]
                ctx.save_for_backward(torch.empty(0))   # nothing but the engine's own refusal of a second pass over a released graph
            with torch.set_grad_enabled(any(ctx.wanted)):
                out = fn(*args)
            ctx.out = out if isinstance(out, tuple) else (out,)
            results = [t.detach() if isinstance(t, torch.Tensor) else t for t in ctx.out]
        results = tuple(_seen(t) for t in results)
        return results if isinstance(out, tuple) else results[0]

    @staticmethod
    def backward(ctx, *grads):
        ctx.saved_tensors
        given = [(t, g) for t, g in zip(ctx.out, grads) if g is not None]
        got = iter(torch.autograd.grad([t for t, _ in given], ctx.inner, [g for _, g in given], retain_graph=True, allow_unused=True)
                   if given else [None] * len(ctx.inner))
        return (None, *[next(got) if want else None for want in ctx.wanted])


def as_one_node(fn):
    """Decorator of a function of positional arguments that calls the native extension: tensors it differentiates are
    arguments of its own, results a tensor or a tuple."""
    @functools.wraps(fn)
    def call(*args):
        return OneNode.apply(fn, *args) if transformed() else fn(*args)
    return call
