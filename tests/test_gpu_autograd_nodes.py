"""Autograd nodes of the native host module where they branch: outputs that nobody uses (their gradient does not arrive), leaf
and non-leaf inputs, and inputs that need no gradient -- against torch autograd on the same operators."""

import pytest
import torch
import torch.nn.functional as F

import cute_kernels

pytestmark = pytest.mark.gpu

# bf16 rounding of inputs to the kernels is shared; results are rounded once to bf16 (2^-9), sums over at most 37 rows in fp32
TOL = dict(rtol=1e-2, atol=2e-2)


def _leaf(shape, g, device):
    return torch.randn(shape, generator=g).to(torch.bfloat16).to(device).requires_grad_()


@pytest.mark.parametrize("used", ["both", "norm", "sum"])
@pytest.mark.parametrize("leaf", [True, False])
def test_residual_add_norm_gradients(device, used, leaf):
    g = torch.Generator().manual_seed(1)
    x, r, w = _leaf((37, 264), g, device), _leaf((37, 264), g, device), _leaf((264,), g, device)
    dy, ds = (torch.randn(37, 264, generator=g).to(torch.bfloat16).to(device) for _ in range(2))
    grads = {}
    for ours in (True, False):
        x.grad = r.grad = w.grad = None
        xi, ri = (x, r) if leaf else (x * 1, r * 1)
        if ours:
            y, s = cute_kernels.fused_residual_add_rmsnorm_cute(xi, ri, w, 1e-6)
        else:
            s = xi + ri
            y = F.rms_norm(s.float(), (264,), w.float(), 1e-6).to(torch.bfloat16)
        outs = [(y, dy), (s, ds)]
        outs = outs if used == "both" else outs[:1] if used == "norm" else outs[1:]
        torch.autograd.backward([o for o, _ in outs], [d for _, d in outs])
        zero = torch.zeros_like(w)
        grads[ours] = [x.grad.clone(), r.grad.clone(), zero if w.grad is None else w.grad.clone()]
        assert x.grad.data_ptr() != r.grad.data_ptr()
    for a, b in zip(grads[True], grads[False]):
        torch.testing.assert_close(a.float(), b.float(), **TOL)


@pytest.mark.parametrize("used", ["rows", "logits"])
def test_norm_route_with_one_output_used(device, used):
    g = torch.Generator().manual_seed(2)
    H, E = 512, 16
    x, nw = _leaf((29, H), g, device), _leaf((H,), g, device)
    gw = (torch.randn(E, H, generator=g) * H**-0.5).to(torch.bfloat16).to(device).requires_grad_()
    dy, dl = torch.randn(29, H, generator=g).to(torch.bfloat16).to(device), torch.randn(29, E, generator=g).to(torch.bfloat16).to(device)
    got = {}
    for ours in (True, False):
        x.grad = nw.grad = gw.grad = None
        if ours:
            y, logits = cute_kernels.rmsnorm_route_cute(x, nw, gw, 1e-6, fused=True)
        else:
            y = F.rms_norm(x.float(), (H,), nw.float(), 1e-6).to(torch.bfloat16)
            logits = F.linear(y, gw)
        (y if used == "rows" else logits).backward(dy if used == "rows" else dl)
        got[ours] = [x.grad.clone(), nw.grad.clone(), None if gw.grad is None else gw.grad.clone()]
    for a, b in zip(got[True], got[False]):
        assert (a is None) == (b is None)
        if a is not None:
            torch.testing.assert_close(a.float(), b.float(), **TOL)


@pytest.mark.parametrize("frozen", ["x", "gate", "c_fc", "c_proj"])
def test_layer_with_a_frozen_part(device, frozen):
    """The gradients that are asked for do not depend on the ones that are not."""
    torch.manual_seed(3)
    moe = cute_kernels.MoE(4, 2, 256, 256, cute_kernels.swiglu_packed_cute, True, False, 256**-0.5).to(torch.bfloat16).to(device)
    x = torch.randn(70, 256, device=device).to(torch.bfloat16).requires_grad_()
    dy = torch.randn(70, 256, device=device).to(torch.bfloat16)
    leaves = {"x": x, "gate": moe.gate.weight, "c_fc": moe.c_fc.weight, "c_proj": moe.c_proj.weight}

    def grads():
        for t in leaves.values():
            t.grad = None
        moe(x)[0].backward(dy)
        return {n: t.grad for n, t in leaves.items()}

    full = grads()
    leaves[frozen].requires_grad_(False)
    part = grads()
    assert part[frozen] is None
    for n in leaves:
        if n != frozen:
            assert torch.equal(part[n], full[n]), n


@pytest.mark.parametrize("grad_mode", [True, False])
def test_forward_mode_is_refused(device, grad_mode):
    """The nodes have no forward-mode rule: a call on a dual tensor raises, whatever the grad mode, and never drops the tangent."""
    x, w = torch.randn(8, 64, device=device), torch.ones(64, device=device)
    calls = [
        lambda d: cute_kernels.rmsnorm_cute(d, w, 1e-6),
        lambda d: cute_kernels.rmsnorm_cute(x, d[0].contiguous(), 1e-6),
        lambda d: cute_kernels.fused_residual_add_rmsnorm_cute(x, d, w, 1e-6),
        lambda d: cute_kernels.swiglu_cute(x, d),
        lambda d: cute_kernels.swiglu_packed_cute(d),
        lambda d: cute_kernels.softmax_cute(d),
        lambda d: cute_kernels.route_topk_softmax(d, 2),
    ]
    with torch.autograd.forward_ad.dual_level(), torch.set_grad_enabled(grad_mode):
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        for call in calls:
            with pytest.raises(RuntimeError, match="jvp"):
                call(dual)


@pytest.mark.parametrize("fn", [cute_kernels.softmax_cute, lambda x: cute_kernels.rmsnorm_cute(x, None, 1e-6)])
def test_rows_without_elements_are_refused(device, fn):
    with pytest.raises(RuntimeError, match="are empty"):
        fn(torch.empty(3, 0, device=device))
