"""Router logits of few rows (ck_router_rows): against float64, with and without the norm ahead, and what keeps the layer's own
gate module."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import cute_kernels
from cute_kernels import _C, rmsnorm_route
from cute_kernels.fp8 import quantize_rows_e4m3

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(B, H, E, dtype):
    g = torch.Generator().manual_seed(B * 7 + H + E)
    x = torch.randn(B, H, generator=g).to(dtype).to(DEV)
    return x, (0.02 * torch.randn(E, H, generator=g)).to(dtype).to(DEV), (1 + 0.1 * torch.randn(H, generator=g)).to(dtype).to(DEV)


def _close_logits(logits, y, w):
    """fp32 sums of H products of 16-bit values, rounded once: off by at most the unit roundoff (2 ** -8 in bf16's 8 bits, 2 ** -11
    in fp16's 11; 2 ** -25 under fp16's smallest normal) and the sum's error, H * 2 ** -24 of the sum of magnitudes."""
    exact = y.double() @ w.double().t().contiguous()
    slack = y.size(1) * 2.0**-24 * (y.double().abs() @ w.double().abs().t().contiguous())
    unit = 2.0**-8 if y.dtype == torch.bfloat16 else 2.0**-11
    assert bool(((logits.double() - exact).abs() <= unit * exact.abs() + (1 + unit) * slack + 2.0**-25).all())


# rows 1, 16, 17: edges of a row block; widths: one piece, an odd number of pieces, 64-column pairs left over, each
# instantiation's largest; experts: one, a ragged block, whole blocks
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,E", [(1, 32, 1), (3, 1024, 8), (16, 1056, 16), (17, 2048, 60), (130, 2080, 128), (33, 4096, 17), (256, 4096, 8)])
def test_logits_and_norm(B, H, E, dtype):
    x, w, nw = _inputs(B, H, E, dtype)
    assert _C.host().router_rows_take(x, w, nw)
    _close_logits(_C.host().router_rows(x, w), x, w)
    for weight in (nw, None):
        y, logits, x8, scale = rmsnorm_route.rmsnorm_route_cute(x, weight, w, 1e-6, quantize=True)
        want = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-6)
        want = want if weight is None else want * weight.double()
        unit = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
        assert bool(((y.double() - want).abs() <= want.abs() * (unit + (1 + unit) * (H + 4) * 2.0**-24) + 2.0**-25).all())
        _close_logits(logits, y, w)
        q, s = quantize_rows_e4m3(y)
        assert torch.equal(x8.view(torch.uint8), q.view(torch.uint8)) and torch.equal(scale, s)


# 4, 8 or 16 rows a workgroup, by how many there are: edges of each, at whole and ragged widths of each instantiation; widths that
# leave whole waves, or half of their pieces, without columns
@pytest.mark.parametrize(
    "B,H,E",
    [(4, 2048, 16), (5, 3072, 33), (500, 1088, 17), (8, 32, 16), (9, 1024, 8), (515, 2016, 32), (1023, 4096, 17), (2049, 992, 1),
     (1030, 2048, 20), (1033, 4064, 32), (3, 256, 8), (17, 512, 33), (2100, 288, 16), (6, 1536, 16), (1000, 1536, 64), (7, 3072, 8)],
)
def test_rows_of_a_workgroup(B, H, E):
    test_logits_and_norm(B, H, E, torch.bfloat16)
    x, w, nw = _inputs(B, H, E, torch.bfloat16)
    w[E // 2, H - 1] = float("inf")  # read again by the pieces past the end of a row: in no other product
    _, logits = rmsnorm_route.rmsnorm_route_cute(x, nw, w, 1e-6)
    assert bool((torch.isfinite(logits).all(0) == (torch.arange(E, device=DEV) != E // 2)).all()) and bool(torch.isinf(logits[:, E // 2]).all())


# 4, 8 and 16 rows a workgroup, at whole and ragged widths
@pytest.mark.parametrize("B,H,E", [(4, 1088, 8), (5, 2048, 8), (600, 1056, 16), (8, 96, 8), (9, 1024, 8), (2050, 992, 8), (2050, 2080, 16)])
def test_rows_whose_squares_vanish(B, H, E):
    """2 ** -80 squared is no fp32 number: without eps the row's reciprocal root is infinite, and so are its values, its logits and its
    e4m3 scale. No NaN out of the columns that a ragged width leaves over."""
    x, w = torch.full((B, H), 2.0**-80, device=DEV, dtype=torch.bfloat16), torch.full((E, H), 0.5, device=DEV, dtype=torch.bfloat16)
    x[1] = 1.0
    y, logits, _, scale = rmsnorm_route.rmsnorm_route_cute(x, None, w, 0.0, quantize=True)
    ordinary = torch.arange(B, device=DEV) == 1
    for t in (y, logits, scale[:, None]):
        assert bool((torch.isinf(t) == ~ordinary[:, None]).all()) and not bool(torch.isnan(t).any())


def test_sizes_beyond_one_workgroup_per_compute_unit_keep_their_routes():
    x, w, _ = _inputs(257, 512, 256, torch.bfloat16)
    take = _C.host().router_rows_take
    assert not take(x, w, None)  # 17 x 16 workgroups
    assert take(x[:256], w, None)
    assert not take(x[:16].float(), w.float(), None)
    assert not take(x[:0], w, None)


def test_rows_off_a_16_byte_boundary_keep_their_routes():
    x, w, nw = _inputs(9, 640, 8, torch.bfloat16)
    off = lambda t: torch.cat([t.new_zeros(3), t.flatten()])[3:].view(t.shape)  # contiguous, 6 bytes past a boundary
    gate = torch.nn.Linear(640, 8, bias=False, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        gate.weight.copy_(w)
        _close_logits(rmsnorm_route.router_logits(gate, off(x)), x, w)
        _close_logits(rmsnorm_route.router_logits(gate, x.t().contiguous().t()), x, w)  # not contiguous: copied
    assert not _C.host().router_rows_take(off(x), w, None)
    assert not _C.host().router_rows_take(x, off(w), None)
    assert not _C.host().router_rows_take(x, w, off(nw))


def test_a_watched_or_replaced_gate_is_called():
    moe = cute_kernels.MoE(8, 2, 512, 256, cute_kernels.swiglu_packed_cute, True, False, 0.02).to(DEV).to(torch.bfloat16)
    x = torch.randn(5, 512, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        plain = moe(x)[1]
        _close_logits(plain, x, moe.gate.weight)
        with torch.autocast("cuda", dtype=torch.float16):
            assert rmsnorm_route.router_logits(moe.gate, x).dtype == torch.float16
        seen = []
        handle = moe.gate.register_forward_hook(lambda m, a, out: seen.append(out))
        moe(x)
        handle.remove()
        assert len(seen) == 1
        moe.gate.forward = lambda rows: torch.zeros(rows.size(0), 8, device=DEV, dtype=rows.dtype)
        assert not moe(x)[1].any()
    del moe.gate.forward
    x.requires_grad_()
    moe(x)[1].float().sum().backward()
    assert x.grad is not None and moe.gate.weight.grad is not None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,E,H", [(1024, 64, 2048), (256, 8, 4096), (1500, 16, 1536), (256, 128, 4096)])
def test_the_same_logits_with_gradients_and_without(T, E, H, dtype):
    """A reentrant checkpoint runs its segment without gradients first and again with them: the same experts have to be selected."""
    x, w, nw = _inputs(T, H, E, dtype)
    gate = torch.nn.Linear(H, E, bias=False, device=DEV, dtype=dtype)
    with torch.no_grad():
        gate.weight.copy_(w)
        plain = rmsnorm_route.router_logits(gate, x)
        y, logits = rmsnorm_route.rmsnorm_route_cute(x, nw, w, 1e-6)
    for leaf in (False, True):
        assert torch.equal(plain, rmsnorm_route.router_logits(gate, x.clone().requires_grad_(leaf)))
        gy, glogits = rmsnorm_route.rmsnorm_route_cute(x.clone().requires_grad_(leaf), nw, gate.weight, 1e-6)
        assert torch.equal(y, gy) and torch.equal(logits, glogits)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("needs", [(True, True), (True, False), (False, True)])
def test_gradients_of_the_few_row_router_are_a_linear_layers(needs, dtype):
    x, w, _ = _inputs(130, 1056, 60, dtype)
    g = torch.randn(130, 60, device=DEV).to(dtype)
    ours, linear = ([t.clone().requires_grad_(n) for t, n in zip((x, w), needs)] for _ in range(2))
    _C.host().router_rows(*ours).backward(g)
    torch.nn.functional.linear(*linear).backward(g)
    for a, b in zip(ours, linear):
        assert (a.grad is None) == (b.grad is None) and (a.grad is None or torch.equal(a.grad, b.grad))


@pytest.mark.parametrize("leaf", [0, 1])
def test_a_leaf_that_no_gradient_is_computed_from_may_be_written_before_the_backward_pass(leaf):
    """As a linear layer has it: the rows' gradient takes the weight only, and the weight's the rows only."""
    x, w, _ = _inputs(33, 640, 8, torch.bfloat16)
    u = torch.randn(33, 8, device=DEV).bfloat16()
    grads = []
    for f in (_C.host().router_rows, torch.nn.functional.linear):
        tensors = [x.clone(), w.clone()]
        tensors[leaf].requires_grad_()
        out = f(*tensors)
        with torch.no_grad():
            tensors[leaf].zero_()
        out.backward(u)
        grads.append(tensors[leaf].grad)
    assert torch.equal(*grads)


def test_second_gradients_and_tangents_of_the_few_row_router():
    x, w, _ = _inputs(33, 640, 8, torch.float16)
    gate = torch.nn.Linear(640, 8, bias=False, device=DEV, dtype=torch.float16)
    gate.weight.data.copy_(w)
    v, u = torch.randn_like(x), torch.randn(33, 8, device=DEV).half()
    seconds = []
    for f in (lambda rows: rmsnorm_route.router_logits(gate, rows), gate):
        leaf, upstream = x.clone().requires_grad_(), u.clone().requires_grad_()
        (first,) = torch.autograd.grad(f(leaf), leaf, upstream, create_graph=True)
        seconds.append(torch.autograd.grad(first, (upstream, gate.weight), v))
    for a, b in zip(*seconds):
        assert torch.equal(a, b)
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():  # a linear layer has a forward-mode rule
        dual = torch.autograd.forward_ad.make_dual(x, v)
        assert torch.autograd.forward_ad.unpack_dual(rmsnorm_route.router_logits(gate, dual)).tangent is not None


def test_backward_hooks_of_the_gate_run():
    gate = torch.nn.Linear(640, 8, bias=False, device=DEV, dtype=torch.bfloat16)
    x = _inputs(9, 640, 8, torch.bfloat16)[0].requires_grad_()
    seen = []
    handles = [gate.register_full_backward_hook(lambda m, gi, go: seen.append("hook")), gate.register_full_backward_pre_hook(lambda m, go: seen.append("pre"))]
    for handle in handles:
        rmsnorm_route.router_logits(gate, x).float().sum().backward()
        handle.remove()
    assert seen == ["pre", "hook", "pre"]
    for register in (torch.nn.modules.module.register_module_full_backward_hook, torch.nn.modules.module.register_module_full_backward_pre_hook):
        handle = register(lambda *a: seen.append("global"))
        rmsnorm_route.router_logits(gate, x).float().sum().backward()
        handle.remove()
    assert seen[3:] == ["global"] * 2


def test_a_router_without_experts_keeps_its_route():
    x, _, nw = _inputs(9, 640, 8, torch.bfloat16)
    w = x.new_empty(0, 640)
    y, logits = rmsnorm_route.rmsnorm_route_cute(x, nw, w, 1e-6)
    assert logits.shape == (9, 0) and torch.equal(y, cute_kernels.rmsnorm_cute(x, nw, 1e-6))


def test_modes_see_the_linear_layer():
    x, w, _ = _inputs(9, 640, 8, torch.bfloat16)
    gate = torch.nn.Linear(640, 8, bias=False, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        gate.weight.copy_(w)
        seen = []

        class Recorder(TorchDispatchMode):
            def __torch_dispatch__(self, func, types, args=(), kwargs=None):
                seen.append(func)
                return func(*args, **(kwargs or {}))

        with Recorder():
            rmsnorm_route.router_logits(gate, x)
        assert torch.ops.aten.mm.default in seen

        class Doubled(torch.overrides.TorchFunctionMode):
            def __torch_function__(self, func, types, args=(), kwargs=None):
                out = func(*args, **(kwargs or {}))
                return 2 * out if func is torch.nn.functional.linear else out

        plain = rmsnorm_route.router_logits(gate, x)
        with Doubled():
            torch.testing.assert_close(rmsnorm_route.router_logits(gate, x), 2 * plain, rtol=2.0**-7, atol=1e-6)
        with torch.device(DEV):  # not a mode that asks for operators
            assert torch.equal(rmsnorm_route.router_logits(gate, x), plain)
