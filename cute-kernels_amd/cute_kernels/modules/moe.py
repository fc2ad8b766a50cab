"""Mixture-of-experts layer with the reference's constructor, sub-module names, state_dict keys and forward contract
(cute_kernels/kernels/scattermoe/torch_implementation.py:12-201; triton_implementation/__init__.py:14-103), running
on the MI355X expert path in cute_kernels.scattermoe."""

from __future__ import annotations

from typing import Callable

import torch
import torch.nn as nn

from .. import _C
from ..scattermoe import (
    _bias_in_epilogue,
    choose_align,
    experts_down,
    experts_up,
    route_topk_softmax,
    route_topk_softmax_raw,
    scattered_experts,
    sort_by_expert,
    swiglu_experts,
)
from ..rmsnorm_route import rmsnorm_route_cute, router_logits
from ..swiglu import swiglu_packed_cute
from ..utils import plain_size


class Experts(nn.Module):
    """One linear layer per expert: weight [num_experts, out_features, in_features], optional bias
    [num_experts, out_features] (torch_implementation.py:12-30,56-60). `forward` takes either of the reference's two call
    forms; both run on the grouped GEMM kernels. (The layer's own `_compute_experts` does not come through here: it fuses
    the two linears and the activation between them.)"""

    def __init__(
        self, num_experts: int, in_features: int, out_features: int, add_bias: bool = True, std: float | None = None
    ) -> None:
        super().__init__()

        self.weight = nn.Parameter(torch.empty(num_experts, out_features, in_features))

        self.bias = None
        if add_bias:
            self.bias = nn.Parameter(torch.empty(num_experts, out_features))

        self.std = std

        self.num_experts = num_experts
        self.in_features = in_features
        self.out_features = out_features

        self.reset_parameters()

    def forward(self, input, *args, **kwargs):
        """Experts_Torch's form (torch_implementation.py:32-49): forward(input, expert_frequency, return_list) with `input`
        the rows grouped by expert ([R, in] or one tensor per expert) -> [R, out] or a list per expert.
        Experts_Triton's form (triton_implementation/__init__.py:14-36): forward(inputs, k, sorted_expert_idxs,
        sorted_scattered_idxs, expert_offsets, gates=None, grouped_in=False, grouped_out=False).
        Told apart by the second argument: a tensor of per-expert row counts, or the integer k. The bias, where the module
        has one, is applied in both forms (the reference's second form drops it)."""
        second = args[0] if args else kwargs.get("expert_frequency", kwargs.get("k"))
        if isinstance(second, torch.Tensor):
            return self._forward_grouped(input, *args, **kwargs)
        return self._forward_scattered(input, *args, **kwargs)

    def _forward_scattered(
        self, inputs, k, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, gates=None, grouped_in=False,
        grouped_out=False,
    ):
        return scattered_experts(
            inputs, self.weight.permute(0, 2, 1), k, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, gates,
            grouped_in, grouped_out, bias=self.bias,
        )

    def _forward_grouped(self, input, expert_frequency: torch.Tensor, return_list: bool):
        if not isinstance(input, torch.Tensor):
            input = torch.cat(list(input))
        rows = input.size(0)
        frequency = expert_frequency.to(torch.long)
        # rows are already grouped: sorted position = row, the expert of a row follows from the counts
        sorted_expert_idxs = torch.repeat_interleave(
            torch.arange(self.num_experts, device=input.device), frequency, output_size=rows
        )
        positions = torch.arange(rows, device=input.device)
        out = scattered_experts(
            input, self.weight.permute(0, 2, 1), 1, sorted_expert_idxs, positions, frequency.cumsum(-1), None, True, True,
            bias=self.bias,
        )
        if return_list:
            out = list(out.split(expert_frequency.tolist(), dim=0))
        return out

    def extra_repr(self):
        return "num_experts={}, in_features={}, out_features={}".format(
            self.num_experts, self.in_features, self.out_features
        )

    @torch.no_grad()
    def reset_parameters(self) -> None:
        nn.init.normal_(self.weight, mean=0, std=self.std)
        if hasattr(self, "bias") and self.bias is not None:
            self.bias.zero_()


class MoE(nn.Module):
    def __init__(
        self,
        num_experts: int,
        num_experts_per_tok: int,
        hidden_size: int,
        intermediate_size: int,
        activation_function: Callable,
        is_glu: bool,
        add_bias: bool,
        std: float,
    ) -> None:
        super().__init__()

        self.num_experts = num_experts
        self.top_k = num_experts_per_tok

        self.hidden_size = hidden_size
        self.intermediate_size = intermediate_size
        self.is_glu = is_glu

        self.gate = nn.Linear(in_features=self.hidden_size, out_features=num_experts, bias=False)

        self.c_fc = Experts(
            num_experts=num_experts,
            in_features=self.hidden_size,
            out_features=2 * self.intermediate_size if is_glu else self.intermediate_size,
            add_bias=add_bias,
            std=std,
        )

        self.act = activation_function

        self.c_proj = Experts(
            num_experts=num_experts,
            in_features=self.intermediate_size,
            out_features=self.hidden_size,
            add_bias=add_bias,
            std=std,
        )

    def forward(self, hidden_states: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
        original_shape = hidden_states.shape

        hidden_states = hidden_states.view(-1, self.hidden_size)
        router_logits, router_weights, selected_experts = self._compute_routing_weights(hidden_states)

        # router_logits -> (total_q, num_experts); router_weights, selected_experts -> (total_q, top_k)
        hidden_states = self._compute_experts(hidden_states, router_weights, selected_experts)
        hidden_states = hidden_states.view(original_shape)

        return hidden_states, router_logits

    def forward_with_norm(
        self, hidden_states: torch.Tensor, norm_weight: torch.Tensor | None, eps: float | None
    ) -> tuple[torch.Tensor, torch.Tensor]:
        """forward(rmsnorm_cute(hidden_states, norm_weight, eps)) with the normalisation fused ahead of the router: one
        kernel reads hidden_states once and writes the normalised rows and the router logits (rmsnorm_route_cute)."""
        original_shape = hidden_states.shape
        normed, router_logits = rmsnorm_route_cute(hidden_states.view(-1, self.hidden_size), norm_weight, self.gate.weight, eps)
        router_weights, selected_experts = route_topk_softmax(router_logits, self.top_k)
        out = self._compute_experts(normed, router_weights.type_as(normed), selected_experts)
        return out.view(original_shape), router_logits

    def _compute_routing_weights(self, hidden_states: torch.Tensor) -> tuple[torch.Tensor]:
        logits = router_logits(self.gate, hidden_states)
        # top-k on the logits and softmax over the k selected logits in fp32, one kernel
        # (torch_implementation.py:127-133); equal logits resolve to the lowest expert index
        router_weights, selected_experts = route_topk_softmax(logits, self.top_k)
        router_weights = router_weights.type_as(hidden_states)
        return logits, router_weights, selected_experts

    def _compute_expert_assignment(
        self, router_weights: torch.Tensor, selected_experts: torch.Tensor
    ) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
        """(fan_in_index [R], batch_gates [R], expert_frequency [E]) as torch_implementation.py:171-193: the token of every
        routed row in expert order (stable: rows of one expert keep their token order), its gate, and the rows per expert
        (int64, like bincount's). One stable counting sort on the GPU instead of bincount + argsort."""
        seg = sort_by_expert(selected_experts.flatten(), self.num_experts)
        order = seg.sorted_scattered_idxs.long()
        fan_in_index = order // self.top_k
        batch_gates = router_weights.flatten()[order]
        return fan_in_index, batch_gates, seg.counts.to(torch.long)

    def _get_topk(self, x: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
        """Top-k values (descending) and int64 indices, as torch_implementation.py:195-201. Not differentiable; the
        layer itself routes through `_compute_routing_weights`."""
        selected, _, values = route_topk_softmax_raw(x, self.top_k)
        return values, selected.long()

    def _needs_grad(self, hidden_states: torch.Tensor, router_weights: torch.Tensor) -> bool:
        """Whether a backward pass may come through the experts. An activation that is the caller's own may hold parameters."""
        if hidden_states.requires_grad or router_weights.requires_grad:
            return True
        if self.act is not swiglu_packed_cute and type(self.act) not in (torch.nn.GLU, torch.nn.GELU):
            return True
        return any(p.requires_grad for p in (*self.c_fc.parameters(), *self.c_proj.parameters()))

    def _compute_experts(
        self, hidden_states: torch.Tensor, router_weights: torch.Tensor, selected_experts: torch.Tensor
    ) -> torch.Tensor:
        if hidden_states.size(0) == 0:  # no tokens: nothing to sort or multiply; the result stays in the autograd graph
            return hidden_states * 0
        inference = not (torch.is_grad_enabled() and self._needs_grad(hidden_states, router_weights))
        align = choose_align(
            plain_size(selected_experts.numel()), self.num_experts, hidden_states.dtype, inference,
            (self.hidden_size, self.intermediate_size, self.is_glu),
        )
        seg = sort_by_expert(selected_experts, self.num_experts, align)
        has_bias = self.c_fc.bias is not None or self.c_proj.bias is not None

        sixteen_bit = hidden_states.dtype != torch.float32  # fp32 layers take the unfused route on the fp32 GEMMs
        if self.is_glu and not has_bias and sixteen_bit:
            # the gated activations this library knows run inside the c_fc epilogue: packed SwiGLU, and torch.nn.GLU over
            # the last dimension (the activation of the reference's own MoE test, tests/test_commons.py:85)
            kind = None
            if self.act is swiglu_packed_cute:
                kind = _C.CK_ACT_SWIGLU
            elif type(self.act) is torch.nn.GLU and self.act.dim in (-1, hidden_states.dim() - 1):
                kind = _C.CK_ACT_GLU
            if kind is not None:
                return swiglu_experts(hidden_states, self.c_fc.weight, self.c_proj.weight, router_weights, seg, kind)

        # any other activation, or expert biases (applied like the reference's torch path, torch_implementation.py:42; its
        # Triton path drops them): grouped GEMM (+ bias) -> activation on the padded grouped rows -> grouped GEMM (+ bias)
        # + gated combine
        if (
            not self.is_glu
            and sixteen_bit
            and type(self.act) is torch.nn.GELU
            and self.act.approximate == "tanh"
            and (self.c_fc.bias is None or _bias_in_epilogue(seg, self.hidden_size))
        ):
            # the non-GLU activation of the reference's layer test (tests/test_commons.py:85-86) runs in the c_fc epilogue
            return experts_up(
                hidden_states, self.c_fc.weight, seg, self.top_k, self.c_fc.bias, gelu_tanh=True,
                down=(self.c_proj.weight, router_weights, self.c_proj.bias),
            )
        hidden_states = experts_up(hidden_states, self.c_fc.weight, seg, self.top_k, self.c_fc.bias)
        hidden_states = self.act(hidden_states)
        hidden_states = experts_down(hidden_states, self.c_proj.weight, router_weights, seg, self.c_proj.bias)
        return hidden_states


# names the reference exports (cute_kernels/kernels/__init__.py:5-21); both resolve to the one implementation here
MoE_Triton = MoE
Experts_Triton = Experts
