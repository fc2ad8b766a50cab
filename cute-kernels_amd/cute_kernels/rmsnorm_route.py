"""RMSNorm fused ahead of the router: y = rmsnorm(x) and router_logits = gate(y) from one pass over x (and, for the
quantised-expert path, the e4m3 rows of y with their scales).

The fused pieces are the reference's rmsnorm forward (cute_kernels/kernels/rmsnorm/triton_implementation/forward.py:14-53,
numerics of F.rms_norm) and the router's linear layer (cute_kernels/kernels/scattermoe/torch_implementation.py:122-124).
Backward: d_y_total = d_y + d_logits @ gate_weight goes through the rmsnorm backward kernel; d_gate_weight = d_logits^T @ y.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F
import torch.nn.modules.module as _module
from torch.utils._device import DeviceContext

from . import _C
from .rmsnorm import rmsnorm_cute
from .utils import is_tracing

MAX_EXPERTS, MAX_HIDDEN, HIDDEN_STEP = 128, 4096, 512


def router_rows_fit(x: torch.Tensor, gate_weight: torch.Tensor, norm_weight: torch.Tensor | None = None) -> bool:
    """Whether few enough 16-bit rows meet few enough experts for the kernel that gives 4 to 16 rows x 16 experts a workgroup of
    their own (ck_router_rows, with or without the norm; the last bits of a token's logits follow how many rows share a
    workgroup, and so the batch). A linear layer casts under autocast. The answer is the same with
    gradients and without: a segment that is checkpointed by running it twice selects the same experts both times."""
    return not is_tracing() and not torch.is_autocast_enabled("cuda") and _C.host().router_rows_take(x, gate_weight, norm_weight)


def _modes_watch() -> bool:
    """Whether a dispatch or function mode (a FLOP counter, a quantiser) is to see the operators that run. The mode behind
    `with torch.device(...)` changes where new tensors live and nothing else."""
    return torch._C._len_torch_dispatch_stack() > 0 or any(
        not isinstance(torch._C._get_function_stack_at(i), DeviceContext) for i in range(torch._C._len_torch_function_stack())
    )


def router_logits(gate: torch.nn.Module, x: torch.Tensor) -> torch.Tensor:
    """gate(x) for rows x [tokens, H]. A plain bias-free nn.Linear that nobody watches (hooks, modes, a forward of its
    own, other tensor types) runs as ck_router_rows on few rows: the library's product takes 15 us there."""
    weight = getattr(gate, "weight", None)
    if (
        not is_tracing()
        and type(gate) is torch.nn.Linear
        and gate.bias is None
        and type(weight) is torch.nn.Parameter
        and type(x) is torch.Tensor
        and x.is_cuda
        and weight.device == x.device
        and weight.dtype == x.dtype
        and x.dim() == 2
        and x.size(1) == weight.size(1)
        and "forward" not in vars(gate)
        and not _modes_watch()
        and not (gate._forward_hooks or gate._forward_pre_hooks or _module._global_forward_hooks or _module._global_forward_pre_hooks)
        and not (gate._backward_hooks or gate._backward_pre_hooks or _module._global_backward_hooks or _module._global_backward_pre_hooks)
        and router_rows_fit(x, weight)
    ):
        return _C.host().router_rows(x, weight)
    return gate(x)


def rmsnorm_route_fused(x: torch.Tensor, gate_weight: torch.Tensor) -> bool:
    """Whether ck_rmsnorm_route takes this shape: 16-bit rows, hidden size a multiple of 512 up to 4096, at most 128 experts.
    Other shapes run rmsnorm_cute followed by the linear layer (and quantize_rows_e4m3), with the same results contract."""
    H, E = x.size(-1), gate_weight.size(0)
    return (
        x.dtype in (torch.bfloat16, torch.float16)
        and H % HIDDEN_STEP == 0
        and H <= MAX_HIDDEN
        and E <= MAX_EXPERTS
        and not is_tracing()
    )


def rmsnorm_route_pays(x: torch.Tensor, gate_weight: torch.Tensor) -> bool:
    """Where the one-pass kernel is the faster route. It re-reads the gate weight from L2 for every 16 rows, so its time
    grows with E * H: 28 us against 40 us for the separate kernels at 8,192 x 2,048 with 64 experts (30 against 53 with the
    e4m3 rows), 62 against 89 at 16,384 x 4,096 with 8. Beyond 64 x 4,096 it pays from
    2,048 rows, where its workgroups begin to fill the chip, up to 16,384. GPU time of 128 experts and rows of 4,096, 513 / 1,024 /
    2,048 / 2,560 / 4,096 / 16,384 of them, one pass 36 / 35 / 36 / 36 / 38 / 90 us, separate 19 / 21 / 28 / 44 / 51 / 113, with the e4m3
    rows 39 / 39 / 40 / 40 / 42 / 122 and 23 / 25 / 33 / 49 / 59 / 139 (65,536 rows: 325 and 321, 436 and 442, a layer 1 % slower); of 96
    experts 1,024 / 2,560 / 4,096 rows 32 / 32 / 34 and 21 / 30 / 49."""
    if gate_weight.size(0) * x.size(-1) <= 64 * 4096:
        return True
    return 2048 * x.size(-1) < x.numel() <= 16384 * x.size(-1)


def rmsnorm_route_cute(
    x: torch.Tensor, norm_weight: torch.Tensor | None, gate_weight: torch.Tensor, eps: float | None, quantize: bool = False,
    fused: bool | None = None,
):
    """(y, router_logits) = (rmsnorm_cute(x, norm_weight, eps), y @ gate_weight^T) with x [..., H] read once; with
    quantize=True (inference) also (x8, scale8) = quantize_rows_e4m3(y): returns (y, router_logits, x8, scale8).

    router_logits [tokens, E] is what `nn.Linear(H, E, bias=False)` with `gate_weight` returns for the 16-bit y (fp32
    accumulation, another summation order: equal within the rounding of the logits' dtype).
    fused: True takes the one-pass kernel wherever it supports the shape, False the separate kernels; None (default)
    ck_router_rows for few rows (router_rows_fit), else the one-pass kernel where it is the faster route
    (rmsnorm_route_pays)."""
    if norm_weight is not None:
        assert norm_weight.dim() == 1 and norm_weight.size(0) == x.size(-1), "hidden size for x and weight tensor is different"
        assert norm_weight.dtype == x.dtype, "tensors weight and y should have same dtype"
    assert gate_weight.dim() == 2 and gate_weight.size(1) == x.size(-1) and gate_weight.dtype == x.dtype, (
        "gate_weight should be [num_experts, hidden_size] in x.dtype"
    )
    if eps is None:
        eps = torch.finfo(x.dtype).eps
    few_rows = fused is None and router_rows_fit(x, gate_weight, norm_weight)
    if fused is None:
        fused = rmsnorm_route_pays(x, gate_weight)
    if few_rows or (fused and rmsnorm_route_fused(x, gate_weight)):
        y, logits, x8, scale8 = _C.host().norm_route(x.reshape(-1, x.size(-1)), norm_weight, gate_weight, eps, quantize, few_rows)
        y = y.view(x.shape)
    else:
        y = rmsnorm_cute(x, norm_weight, eps)
        logits = F.linear(y.view(-1, y.size(-1)), gate_weight)
        x8 = scale8 = None
        if quantize:
            from .fp8 import quantize_rows_e4m3

            x8, scale8 = quantize_rows_e4m3(y.detach().view(-1, y.size(-1)))
    return (y, logits, x8, scale8) if quantize else (y, logits)
