"""Forward-only guard of the module layer.

The kernels compute the inference forward pass: no dropout mask is drawn (the reference's
DropoutRowwise / DropoutColumnwise are the identity only in eval mode, dropout.py:57-58) and no
autograd graph is recorded.  A call that expects either must fail instead of silently returning
an un-dropped, non-differentiable result.
"""
from __future__ import annotations

import functools

import torch


def _wants_gradient(values):
    for v in values:
        if isinstance(v, torch.Tensor):
            if v.requires_grad:
                return True
        elif isinstance(v, (list, tuple)) and _wants_gradient(v):
            return True
    return False


def refuse_training(module, args=(), kwargs=None):
    """Raises RuntimeError when `module` is in training mode, or when autograd is recording and an
    input tensor asks for a gradient."""
    if module.training:
        raise RuntimeError(
            "%s is forward-only (inference): call .eval() first.  In training mode the reference applies "
            "dropout and records gradients; these kernels do neither." % type(module).__name__)
    if torch.is_grad_enabled() and (_wants_gradient(args) or (kwargs and _wants_gradient(kwargs.values()))):
        raise RuntimeError(
            "%s is forward-only (inference): an input requires a gradient, and the kernels record no "
            "autograd graph.  Detach the input or call under torch.no_grad()." % type(module).__name__)


def forward_only(fn):
    """Method decorator: refuse_training(self, inputs), then run under torch.no_grad()."""

    @functools.wraps(fn)
    def wrapper(self, *args, **kwargs):
        refuse_training(self, args, kwargs)
        with torch.no_grad():
            return fn(self, *args, **kwargs)

    return wrapper
