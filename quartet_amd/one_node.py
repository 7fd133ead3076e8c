"""The native layer calls as one autograd node of Python, for callers that record or transform what Python runs.

The layers' autograd functions are native (csrc/host_ext.cpp): what they allocate goes through PyTorch's operators, what
they launch does not.  ``torch.jit.trace`` would therefore record the allocations and leave the launches out, and a replay
would return memory nobody wrote.  Under a trace a call goes through a Python autograd function instead, which the
trace keeps as one node that runs the whole call again: packed weights are looked up, and random numbers drawn, on every
replay."""
import functools

import torch


def transformed():
    """Whether the calls of this thread are being recorded by a trace."""
    return torch.jit.is_tracing()


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
        return _OneNode.apply(fn, *args) if transformed() else fn(*args)
    return call
