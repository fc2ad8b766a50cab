"""SwiGLU: `up * gate * sigmoid(gate)`, separate and packed ([up | gate] along the last dim).

API and autograd mirror cute_kernels/kernels/swiglu/__init__.py:74-175 (reference).
"""

from __future__ import annotations

import torch

from . import _C
from .utils import divide_if_divisible, is_tracing

_ops = None  # cute_kernels.compile_ops, set by the package once it is imported (used only while torch.compile traces)


def swiglu_cute(
    gate: torch.Tensor,
    up: torch.Tensor,
    *,
    kernel_backend_forward=None,
    kernel_backend_backward=None,
) -> torch.Tensor:
    """computes swiglu activation as `up` * `gate` * sigmoid(`gate`)

    Args:
        gate (torch.Tensor): `gate` activation tensor
        up (torch.Tensor): `up` activation tensor
        kernel_backend_forward, kernel_backend_backward: accepted for call compatibility with the reference and
            ignored -- there is one backend here (HIP on gfx950).

    Returns:
        torch.Tensor: output tensor
    """
    assert gate.size() == up.size(), "tensors gate and up should have same shape"
    assert gate.dtype == up.dtype and gate.device == up.device, "tensors gate and up should have same dtype"
    if is_tracing():
        return _ops.swiglu(gate, up)
    return _C.host().swiglu(gate, up)


def swiglu_packed_cute(x: torch.Tensor) -> torch.Tensor:
    """computes swiglu activation by splitting the tensor `x` into 2 parts along the last dim: up (first half) and
    gate (second half)

    Args:
        x (torch.Tensor): input activation

    Returns:
        torch.Tensor: output tensor
    """
    divide_if_divisible(x.size(-1), 2)
    if is_tracing():
        return _ops.swiglu_packed(x)
    return _C.host().swiglu_packed(x)
