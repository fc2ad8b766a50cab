"""Layers in the modes that share the inference heights: under no_grad, compiled under no_grad, and with nothing to differentiate."""

import pytest
import torch

import cute_kernels as ck

pytestmark = pytest.mark.gpu


@pytest.mark.timeout(300)
@pytest.mark.parametrize("act,bias", [("swiglu", False), ("gelu", True), ("silu", True)])
@pytest.mark.parametrize("rows", [4, 12, 20, 40])  # tiles of 16, 32, 64 and 128 rows
def test_same_kernels_in_every_inference_mode(device, act, bias, rows):
    torch.manual_seed(rows)
    E, H, I = 8, 256, 320
    fn, gated = {"swiglu": (ck.swiglu_packed_cute, True), "gelu": (torch.nn.GELU("tanh"), False), "silu": (torch.nn.SiLU(), False)}[act]
    moe = ck.MoE(E, 2, H, I, fn, gated, bias, 0.05).to(device, torch.bfloat16)
    if bias:
        with torch.no_grad():
            moe.c_fc.bias.normal_(0, 0.1)
            moe.c_proj.bias.normal_(0, 0.1)
    x = torch.randn(rows * E // 2, H, device=device).to(torch.bfloat16)
    trained = moe(x)[0].detach()
    torch._dynamo.reset()
    compiled = torch.compile(moe, fullgraph=True, backend="aot_eager", dynamic=False)
    with torch.no_grad():
        want = moe(x)[0]
        assert torch.equal(compiled(x)[0], want)
    # the training forward sums the same fp32 products in another order: one rounding step of bf16 apart, on outputs of O(0.1)
    torch.testing.assert_close(want.float(), trained.float(), rtol=1e-2, atol=1e-2)
    moe.requires_grad_(False)
    frozen = moe(x)[0]
    if act == "silu":  # an activation that the layer does not know: the heights of training
        assert torch.equal(frozen, trained)
    else:
        assert torch.equal(frozen, want)


@pytest.mark.parametrize("rows,height", [(40, 128), (300, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_expert_linear_on_both_heights(device, monkeypatch, dtype, rows, height):
    """ck.Experts forward and backward against one matrix product per expert in fp32."""
    E, K, N = 32, 512, 512
    torch.manual_seed(rows)
    seen, real = [], ck.scattermoe.segments_from_sorted
    monkeypatch.setattr(ck.scattermoe, "segments_from_sorted", lambda *a: (seen.append(a[3]), real(*a))[1])
    experts = ck.Experts(E, K, N, False, K**-0.5).to(device, dtype)
    counts = torch.full((E,), rows, device=device)
    x = torch.randn(rows * E, K, device=device).to(dtype).requires_grad_()
    dy = torch.randn(rows * E, N, device=device).to(dtype)
    y = experts(x, counts, return_list=False)
    y.backward(dy)
    assert set(seen) == {height if dtype is torch.bfloat16 else 128}
    w, xr = experts.weight.detach().float(), x.detach().float().view(E, rows, K)
    tol = dict(rtol=1e-2, atol=2e-2) if dtype is torch.bfloat16 else dict(rtol=1e-4, atol=1e-4)  # O(1) results; dW below: O(sqrt(rows))
    torch.testing.assert_close(y.detach().float().view(E, rows, N), torch.bmm(xr, w.transpose(1, 2).contiguous()), **tol)
    dyr = dy.float().view(E, rows, N)
    torch.testing.assert_close(x.grad.float().view(E, rows, K), torch.bmm(dyr, w), **tol)
    want = torch.bmm(dyr.transpose(1, 2).contiguous(), xr)
    torch.testing.assert_close(experts.weight.grad.float() / rows**0.5, want / rows**0.5, **tol)
