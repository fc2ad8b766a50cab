"""The tanh-GELU layer as one autograd node: its grouped rows have pads that nothing writes, and nobody outside may see them."""

import pytest
import torch

import cute_kernels
from cute_kernels import scattermoe

pytestmark = pytest.mark.gpu


def _layer(device, bias):
    torch.manual_seed(4)
    moe = cute_kernels.MoE(5, 2, 256, 520, torch.nn.GELU(approximate="tanh"), False, bias, 0.05).to(torch.float16).to(device)
    if bias:
        with torch.no_grad():
            moe.c_fc.bias.normal_(0, 0.1)
            moe.c_proj.bias.normal_(0, 0.1)
    x = torch.randn(90, 256, device=device).to(torch.float16).requires_grad_()
    return moe, x, torch.randn(90, 256, device=device).to(torch.float16)


def _grads(moe, x, dy):
    leaves = {"x": x, **dict(moe.named_parameters())}
    for t in leaves.values():
        t.grad = None
    moe(x)[0].backward(dy)
    return {n: t.grad for n, t in leaves.items()}


@pytest.mark.parametrize("bias", [False, True])
def test_anomaly_mode_finds_nothing(device, bias):
    """With new memory filled with NaN (what deterministic mode does) and every node's gradients checked for it."""
    moe, x, dy = _layer(device, bias)
    want = _grads(moe, x, dy)
    torch.use_deterministic_algorithms(True, warn_only=True)
    try:
        with torch.autograd.detect_anomaly(check_nan=True):
            got = _grads(moe, x, dy)
    finally:
        torch.use_deterministic_algorithms(False)
    for n in want:
        assert torch.equal(want[n], got[n]), n


@pytest.mark.parametrize("frozen", [(), ("x",), ("c_fc.weight", "c_fc.bias"), ("x", "c_fc.weight", "c_fc.bias"), ("gate.weight",),
                                    ("c_proj.weight", "c_proj.bias"), ("x", "c_fc.weight", "c_proj.weight")])
def test_same_gradients_as_two_linears(device, frozen):
    """The node against experts_up and experts_down (the same kernels in the same order), with parts that need no gradient."""
    moe, x, dy = _layer(device, True)
    params = {"x": x, **dict(moe.named_parameters())}
    for n in frozen:
        params[n].requires_grad_(False)
    with torch.no_grad():
        gates, ids = scattermoe.route_topk_softmax(moe.gate(x), 2)
    seg = cute_kernels.sort_by_expert(ids, 5, 256)
    res = []
    for node in (True, False):
        gates = gates.detach().requires_grad_("gate.weight" not in frozen)
        for t in params.values():
            t.grad = None
        fc, proj = moe.c_fc, moe.c_proj
        if node:
            y = scattermoe.experts_up(x, fc.weight, seg, 2, fc.bias, gelu_tanh=True, down=(proj.weight, gates, proj.bias))
        else:
            y = scattermoe.experts_down(scattermoe.experts_up(x, fc.weight, seg, 2, fc.bias, gelu_tanh=True), proj.weight, gates, seg, proj.bias)
        y.backward(dy)
        res.append([y.detach(), gates.grad] + [t.grad for t in params.values()])
    for a, b in zip(*res):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))
