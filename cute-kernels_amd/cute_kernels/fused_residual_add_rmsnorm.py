"""Residual add fused with RMSNorm: (x * multiplier + residual) -> (rmsnorm of the sum, the sum).

API and autograd mirror cute_kernels/kernels/fused_residual_add_rmsnorm/__init__.py:15-108 (reference); numerics follow
fused_residual_add_rmsnorm_torch (torch_implementation.py:9-19): the scaled x and the sum are each rounded to the tensor
dtype before the norm, which itself follows F.rms_norm.
"""

from __future__ import annotations

import torch

from . import _C
from .utils import is_tracing

_ops = None  # cute_kernels.compile_ops, set by the package once it is imported (used only while torch.compile traces)


def fused_residual_add_rmsnorm_cute(
    x: torch.Tensor,
    residual: torch.Tensor,
    weight: torch.Tensor | None,
    eps: float | None,
    multiplier: float | None = None,
    memory_efficient: bool = False,
) -> tuple[torch.Tensor, torch.Tensor]:
    """fused residual add RMSNorm computation

    Args:
        x (torch.Tensor): input activation
        residual (torch.Tensor): residual activation
        weight (torch.Tensor | None): RMSNorm weight
        eps (float | None): epsilon; None uses torch.finfo(x.dtype).eps
        multiplier (float | None, optional): if not None, pre-multiplies `x` with `multiplier`. Defaults to None.
        memory_efficient (bool, optional): memory efficient = False caches RMSNorm's denominator in the forward.
            Defaults to False.

    Returns:
        tuple[torch.Tensor, torch.Tensor]: output activations, updated residual stream
    """
    if weight is not None:
        assert weight.dim() == 1, "weight should be 1D"
        assert weight.size(-1) == x.size(-1), "hidden size for x and weight tensor is different"
        assert weight.dtype == x.dtype and weight.device == x.device, "tensors weight and y should have same dtype"
    assert residual.shape == x.shape and residual.dtype == x.dtype, "x and residual should match"
    if eps is None:
        eps = torch.finfo(x.dtype).eps
    multiplier = 1.0 if multiplier is None else float(multiplier)
    if is_tracing():
        output, added_x_residual, _ = _ops.fused_residual_add_rmsnorm(x, residual, weight, eps, multiplier, memory_efficient)
        return output, added_x_residual
    return _C.host().residual_rmsnorm(x, residual, weight, eps, multiplier, memory_efficient)
