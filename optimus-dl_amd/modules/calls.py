"""How the modules call what a graph compiler must not trace, and autograd functions that nothing will differentiate.

Both are about host time: an evaluation step of a few tokens waits for the host, not for the GPU.  The wrapper of
``torch.compiler.disable`` costs about 3 us a call and ``Function.apply`` about 8, of some 25 per kernel of such a step.
"""

from __future__ import annotations

import functools

import torch
import torch.autograd.forward_ad as _forward_ad

# Whether a graph compiler, a functorch transform, forward-mode differentiation or a tracer is at work is known to private
# parts of torch only.  Where a version of torch lacks one of them, every call takes the long way.
try:
    from torch._C._dynamo.eval_frame import get_eval_frame_callback as _compiler_callback
except ImportError:
    def _compiler_callback():
        return False

_functorch_stack = getattr(getattr(torch._C, "_functorch", None), "peek_interpreter_stack", None)
_tracing_state = getattr(torch._C, "_get_tracing_state", None)
_graph_state_known = _functorch_stack is not None and _tracing_state is not None and hasattr(_forward_ad, "_current_level")


def untraced(fn):
    """``torch.compiler.disable(fn)``, without its wrapper where no graph compiler is at work on this thread."""
    disabled = torch.compiler.disable(fn)

    @functools.wraps(fn)
    def call(*args, **kwargs):
        if torch.compiler.is_compiling() or _compiler_callback() is not None:
            return disabled(*args, **kwargs)
        return fn(*args, **kwargs)

    return call


class _NoGraph:
    """The context of a forward that leaves no node behind."""

    def __init__(self, n: int):
        self.needs_input_grad = (False,) * n

    def save_for_backward(self, *tensors: torch.Tensor) -> None:
        pass

    # what else a forward may tell its context is about the node
    mark_dirty = mark_non_differentiable = save_for_forward = save_for_backward

    def set_materialize_grads(self, value: bool) -> None:
        pass


def no_graph() -> bool:
    """Whether nothing records, transforms or traces what runs now."""
    return not (not _graph_state_known or torch.is_grad_enabled() or _forward_ad._current_level >= 0 or _functorch_stack() is not None
                or _tracing_state() is not None)


def apply(function: "type[torch.autograd.Function]", *args):
    """``function.apply(*args)``; only its forward where no graph is recorded.

    ``Function.apply`` reports parameters that require gradients as needing one also under ``torch.no_grad()``: a forward
    that prepares operands of the backward (transposed codes) would make them for nobody.  Whatever else looks at an
    autograd function still finds it: functorch transforms, forward-mode differentiation and the tracer of torch.jit."""
    if not no_graph():
        return function.apply(*args)
    return function.forward(_NoGraph(len(args)), *args)
