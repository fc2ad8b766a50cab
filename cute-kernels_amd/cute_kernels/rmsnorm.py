"""RMSNorm forward / backward.

API and autograd mirror cute_kernels/kernels/rmsnorm/__init__.py:12-77 (reference); numerics follow F.rms_norm, the
reference's oracle (rmsnorm/torch_implementation.py:9-10).
"""

from __future__ import annotations

import torch

from . import _C
from .utils import is_tracing

_ops = None  # cute_kernels.compile_ops, set by the package once it is imported (used only while torch.compile traces)


def rmsnorm_cute(
    x: torch.Tensor, weight: torch.Tensor | None, eps: float | None, memory_efficient: bool = False
) -> torch.Tensor:
    """RMSNorm computation

    Args:
        x (torch.Tensor): input activation
        weight (torch.Tensor | None): RMSNorm weight
        eps (float | None): epsilon; None uses torch.finfo(x.dtype).eps
        memory_efficient (bool, optional): memory efficient = False caches RMSNorm's denominator in the forward.
            Defaults to False.

    Returns:
        torch.Tensor: output tensor
    """
    if weight is not None:
        assert weight.dim() == 1, "weight should be 1D"
        assert weight.size(-1) == x.size(-1), "hidden size for x and weight tensor is different"
        assert weight.dtype == x.dtype and weight.device == x.device, "tensors weight and y should have same dtype"
    if eps is None:
        eps = torch.finfo(x.dtype).eps
    if is_tracing():
        return _ops.rmsnorm(x, weight, eps, memory_efficient)[0]
    return _C.host().rmsnorm(x, weight, eps, memory_efficient)
