"""Softmax over the last dimension, with an optional logits multiplier.

API and autograd mirror cute_kernels/kernels/softmax/__init__.py:12-50 (reference); numerics follow softmax_torch
(softmax/torch_implementation.py:9-18): fp32 math, result cast back to the input dtype.
"""

from __future__ import annotations

import torch

from . import _C
from .utils import is_tracing

_ops = None  # cute_kernels.compile_ops, set by the package once it is imported (used only while torch.compile traces)


def softmax_cute(x: torch.Tensor, logits_multiplier: float | None = None) -> torch.Tensor:
    """computes softmax activation

    Args:
        x (torch.Tensor): input activation tensor
        logits_multiplier (float, optional): pre-multiplies `x` with `logits_multiplier` before computing softmax.
            Defaults to None.

    Returns:
        torch.Tensor: output tensor
    """
    multiplier = 1.0 if logits_multiplier is None else float(logits_multiplier)
    if is_tracing():
        return _ops.softmax(x, multiplier)
    return _C.host().softmax(x, multiplier)
