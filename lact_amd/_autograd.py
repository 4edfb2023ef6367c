"""What the autograd functions of this package share."""
from __future__ import annotations

import functools

import torch

from . import _lib


def once_differentiable(backward):
    """torch.autograd.function.once_differentiable without its gaps: that one refuses a second derivative only where the incoming
    gradients depend on something, and only when the whole graph is walked.  The results here depend on the saved tensors, and an
    error on every path from them to the function's inputs says that this dependence cannot be followed."""
    @functools.wraps(backward)
    def wrapper(ctx, *grads):
        with torch.no_grad():
            res = backward(ctx, *grads)
        if not torch.is_grad_enabled():
            return res
        refused = _lib.host().refuse_second_derivative(list(res) if isinstance(res, tuple) else [res])
        return tuple(refused) if isinstance(res, tuple) else refused[0]
    return wrapper
