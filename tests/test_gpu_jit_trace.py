"""torch.jit.trace records the operators, not the tensors that eager launches would write past it."""

import pytest
import torch

import cute_kernels as ck

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore")]

H = 64
CALLS = {
    "rmsnorm": (1, lambda x, w: ck.rmsnorm_cute(x, w, 1e-6)),
    "residual": (2, lambda x, r, w: ck.fused_residual_add_rmsnorm_cute(x, r, w, 1e-6)),
    "swiglu": (2, lambda x, u, w: ck.swiglu_cute(x, u)),
    "swiglu_packed": (1, lambda x, w: ck.swiglu_packed_cute(x)),
    "softmax": (1, lambda x, w: ck.softmax_cute(x, 0.5)),
    "route": (1, lambda x, w: ck.route_topk_softmax(x, 2)[0]),
}


def _check(fn, make):
    """A trace made with one set of inputs, run on another, against the eager call: outputs and gradients bit for bit."""
    traced = torch.jit.trace(fn, make(), check_trace=False)
    inputs = make()
    results = []
    for call in (traced, fn):
        outs = call(*inputs)
        outs = outs if isinstance(outs, tuple) else (outs,)
        total = sum(t.float().square().sum() for t in outs)
        results.append([*outs, *torch.autograd.grad(total, inputs)])
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("name", list(CALLS))
def test_operators(device, name):
    n, fn = CALLS[name]
    w = torch.rand(H, device=device)
    _check(lambda *a: fn(*a, w), lambda: tuple(torch.randn(9, H, device=device, requires_grad=True) for _ in range(n)))


@pytest.mark.parametrize("tokens", [8, 2200])
def test_layer(device, tokens):
    torch.manual_seed(1)
    moe = ck.MoE(4, 2, H, 64, ck.swiglu_packed_cute, True, False, 0.1).to(device, torch.bfloat16)
    moe.gate.weight.requires_grad_(False)  # the router's share of the gradient passes through d_gates in 16 bits in a trace
    make = lambda: torch.randn(tokens, H, device=device).to(torch.bfloat16)
    traced = torch.jit.trace(moe, (make(),), check_trace=False)
    x = make()
    results = []
    for call in (traced, moe):
        moe.zero_grad(set_to_none=True)
        y, logits = call(x)
        y.float().square().sum().backward()
        results.append([y, logits, moe.c_fc.weight.grad, moe.c_proj.weight.grad])
    for a, b in zip(*results):
        assert torch.equal(a, b)
