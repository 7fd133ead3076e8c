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
from torch._C import _are_functorch_transforms_active, _is_tracing   # 0.15 us a call together; through torch.jit 0.3
from torch.autograd import forward_ad


def transformed():
    """Whether calls are being recorded by a trace, carry forward-mode tangents or run inside a ``torch.func`` transform."""
    return _is_tracing() or forward_ad._current_level >= 0 or _are_functorch_transforms_active()


class _OneNode(torch.autograd.Function):
    """fn(*args) with the native graph behind its outputs kept inside the node."""

    @staticmethod
    def forward(ctx, fn, *args):
        ctx.set_materialize_grads(False)
        ctx.wanted = ctx.needs_input_grad[1:]
        if not any(ctx.wanted):
            return fn(*args)
        inner = [a.detach().requires_grad_(want) if isinstance(a, torch.Tensor) else a for a, want in zip(args, ctx.wanted)]
        with torch.enable_grad():
            out = fn(*inner)
        ctx.inner = [a for a, want in zip(inner, ctx.wanted) if want]
        ctx.out = out if isinstance(out, tuple) else (out,)
        ctx.save_for_backward(torch.empty(0))   # nothing but the engine's own refusal of a second pass over a released graph
        detached = tuple(t.detach() if isinstance(t, torch.Tensor) else t for t in ctx.out)
        return detached if isinstance(out, tuple) else detached[0]

    @staticmethod
    def backward(ctx, *grads):
        ctx.saved_tensors
        given = [(t, g) for t, g in zip(ctx.out, grads) if g is not None]
        got = iter(torch.autograd.grad([t for t, _ in given], ctx.inner, [g for _, g in given], retain_graph=True, allow_unused=True)
                   if given else [None] * len(ctx.inner))
        return (None, *[next(got) if want else None for want in ctx.wanted])


def one_node(fn):
    """Decorator of a function of positional arguments that calls the native extension: tensors it differentiates are
    arguments of its own, results a tensor or a tuple."""
    @functools.wraps(fn)
    def call(*args):
        if _is_tracing() or forward_ad._current_level >= 0 or _are_functorch_transforms_active():   # transformed(), without its call
            return _OneNode.apply(fn, *args)
        return fn(*args)
    return call
