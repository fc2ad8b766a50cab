"""Saved-tensor hooks over the layers' nodes: they see the tensors that a user knows, and what they hand back is used."""

import pytest
import torch

import cute_kernels as ck

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["swiglu", "gelu", "silu"])
def test_hooks_that_compress_or_move(device, act):
    fn, gated = {"swiglu": (ck.swiglu_packed_cute, True), "gelu": (torch.nn.GELU("tanh"), False), "silu": (torch.nn.SiLU(), False)}[act]
    torch.manual_seed(2)
    moe = ck.MoE(4, 2, 256, 256, fn, gated, not gated, 0.05).to(device, torch.bfloat16)
    x = torch.randn(70, 256, device=device).to(torch.bfloat16).requires_grad_()
    dy = torch.randn(70, 256, device=device).to(torch.bfloat16)
    leaves = [x, *moe.parameters()]
    seen = []

    def pack(t):  # exact for 16-bit tensors and for whole numbers up to 2^24
        seen.append(t.dtype)
        t.abs().max()  # as a quantising hook would; there is none for unsigned words
        return t.float().cpu(), t.dtype

    hooks = {
        "none": None,
        "own": torch.autograd.graph.saved_tensors_hooks(pack, lambda p: p[0].to(device).to(p[1])),
        "cpu": torch.autograd.graph.save_on_cpu(pin_memory=True),
    }
    grads = {}
    for name, hook in hooks.items():
        for t in leaves:
            t.grad = None
        if hook is None:
            y = moe(x)[0]
        else:
            with hook:
                y = moe(x)[0]
        y.backward(dy)
        grads[name] = [t.grad for t in leaves]
    assert torch.uint32 not in seen and torch.bfloat16 in seen
    for name in ("own", "cpu"):
        for a, b in zip(grads[name], grads["none"]):
            assert torch.equal(a, b), name
