"""Which tile height a call gets (scattermoe.choose_align): one rule for the eager layer, the traced one and the reference's
expert-linear interface. Nothing is launched; traced calls end at the first real operator, which refuses the CPU tensor."""

import math
import sys

import pytest
import torch

import cute_kernels as ck
from cute_kernels import scattermoe
from cute_kernels.modules import moe as moe_module

BF16 = torch.bfloat16
E = 8


def _layer(act="swiglu", H=256, I=320, dtype=BF16):
    fn, gated = {"swiglu": (ck.swiglu_packed_cute, True), "gelu": (torch.nn.GELU("tanh"), False), "silu": (torch.nn.SiLU(), False),
                 "prelu": (torch.nn.PReLU(), False)}[act]
    return ck.MoE(E, 2, H, I, fn, gated, False, 0.02).to(dtype)


class _Stop(Exception):
    pass


def _eager_align(monkeypatch, moe, rows, grad):
    """the height the eager layer sorts with"""
    seen = []
    monkeypatch.setattr(moe_module, "route_topk_softmax", lambda x, k, **kw: (x.softmax(-1).topk(k)[0], x.topk(k)[1]))

    def sort(ids, experts, align=None):
        seen.append(align)
        raise _Stop

    monkeypatch.setattr(moe_module, "sort_by_expert", sort)
    with torch.set_grad_enabled(grad), pytest.raises(_Stop):
        moe(torch.randn(rows * E // 2, moe.hidden_size, dtype=moe.gate.weight.dtype))
    return seen[0]


class _Backend:
    """Keeps the `align` argument of every sort (or of every expert linear) in the graphs it is given."""

    def __init__(self):
        self.aligns, self.graphs = [], 0

    def __call__(self, gm, inputs):
        self.graphs += 1
        ops = torch.ops.ck_mi355
        for n in gm.graph.nodes:
            if n.target in (ops.sort_by_expert, ops.sort_by_expert.default):
                self.aligns.append(n.args[2])
            if n.target in (ops.scattered_experts, ops.scattered_experts.default):
                self.aligns.append(n.args[10])
        return gm.forward


def _traced(fn, x, backend, grad, **kw):
    torch._dynamo.reset()
    compiled = torch.compile(fn, fullgraph=True, backend=backend, **kw)
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError, match="runs on the GPU only"):
        compiled(x)
    return compiled


def test_a_caller_that_says_only_the_sizes():
    for dtype, inference, widths in ((None, False, None), (torch.float32, True, (256, 320, True)), (torch.float32, False, (4096, 14336, True))):
        for rows in (1, 40, 192, 511):
            assert scattermoe.choose_align(rows * E, E, dtype, inference, widths) == 128
        assert scattermoe.choose_align(512 * E, E, dtype, inference, widths) == 256


def test_the_quantised_layer_never_gets_128_rows():
    aligns = [scattermoe.choose_align(rows * E, E, BF16, inference=True) for rows in range(1, 600)]
    assert set(aligns) == {16, 32, 64, 256}


@pytest.mark.parametrize("H,I,gated,rows,training,height", [
    (4096, 14336, True, 8, True, 256), (4096, 14336, True, 400, True, 256), (1024, 1024, True, 96, True, 128),
    (3200, 1120, True, 32, True, 128), (3200, 1120, True, 400, True, 256), (1024, 1024, False, 16, True, 128),
    (4096, 14336, True, 128, False, 256), (1664, 5632, True, 40, False, 128), (1664, 5632, True, 300, False, 256),
])
def test_sixteen_bit_layers_take_the_faster_height(H, I, gated, rows, training, height):
    """8 experts, far from where the two heights meet (the times beside the rule: 1.15 to 2.7 times apart)."""
    assert scattermoe.choose_align(rows * E, E, BF16, not training, (H, I, gated)) == height


@pytest.mark.parametrize("experts,H,I,gated,rows", [(8, 2048, 4096, False, 160), (8, 2048, 4096, False, 230), (16, 1024, 2016, True, 16),
                                                    (16, 1024, 2016, True, 64), (8, 1024, 3840, True, 40)])
def test_a_split_last_round_makes_up_for_its_exchange(experts, H, I, gated, rows):
    """Training steps of few tiles whose long launches split their last round on 256 rows: 128 rows are 1.11 to 1.34 times slower (498,
    617, 307, 359 and 363 against 401, 461, 276, 312 and 275 us)."""
    assert scattermoe.choose_align(rows * experts, experts, BF16, False, (H, I, gated)) == 256


@pytest.mark.parametrize("experts,columns,contraction,rows,grad,height", [
    (16, 4576, 3072, 289, False, 256), (32, 3840, 3904, 51, False, 256), (64, 2784, 4096, 14, False, 256), (32, 1600, 672, 244, False, 128),
    (8, 4352, 2240, 28, True, 256), (16, 3072, 832, 211, True, 256), (8, 1664, 3840, 36, True, 256), (8, 1024, 1024, 96, True, 128),
    (32, 512, 512, 300, True, 256), (32, 512, 512, 40, True, 128),
])
def test_single_linears_take_the_faster_height(experts, columns, contraction, rows, grad, height):
    """scattered_experts, forward alone and with its backward: 230, 254, 332, 49, 229, 175, 152 us with the other height, 193, 195, 267, 39,
    167, 153, 131 with this one; 32 x 512 x 512 at 300 rows 71 and 70 (Zipf(0.8): 93 and 90), at 40 rows 52 and 48."""
    launches = ((columns, contraction, False),) + (((contraction, columns, True),) if grad else ())
    assert scattermoe._large_tiles(rows * experts, experts, BF16, not grad, launches, False) == height


@pytest.mark.parametrize("act", ["swiglu", "gelu", "silu", "prelu"])
@pytest.mark.parametrize("rows", [4, 40, 200, 600])
def test_nothing_to_differentiate_is_inference(monkeypatch, act, rows):
    """Gradients enabled, but no tensor asks for one: the inference heights, except where the activation is a callable that
    may hold parameters (its output then needs a gradient, which the small tiles' GEMMs do not have)."""
    moe = _layer(act)
    want = {grad: _eager_align(monkeypatch, moe, rows, grad) for grad in (False, True)}
    for p in moe.parameters():
        p.requires_grad_(False)
    if act == "prelu":
        moe.act.weight.requires_grad_(True)
    assert _eager_align(monkeypatch, moe, rows, True) == want[act in ("silu", "prelu")]
    assert _eager_align(monkeypatch, moe, rows, False) == want[False]


@pytest.mark.parametrize("act", ["swiglu", "gelu", "silu"])
@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("rows", [4, 20, 40, 200, 600])
def test_the_traced_layer_takes_the_eager_height(monkeypatch, act, grad, rows):
    moe, backend = _layer(act), _Backend()
    _traced(lambda x: moe(x)[0], torch.randn(rows * E // 2, moe.hidden_size, dtype=BF16), backend, grad, dynamic=False)
    assert backend.aligns == [_eager_align(monkeypatch, moe, rows, grad)]


@pytest.mark.parametrize("grad", [False, True])
def test_a_dynamic_row_count_compiles_two_graphs(grad):
    """128 rows below 512 rows per expert, 256 from there on, and not a graph for every line of the rule."""
    moe, backend = _layer(), _Backend()
    shapes = [rows * E // 2 for rows in (4, 10, 20, 40, 120, 300, 511, 512, 700, 2000)]
    compiled = _traced(lambda x: moe(x)[0], torch.randn(shapes[0], 256, dtype=BF16), backend, grad, dynamic=True)
    for T in shapes[1:]:
        with torch.set_grad_enabled(grad), pytest.raises(RuntimeError, match="runs on the GPU only"):
            compiled(torch.randn(T, 256, dtype=BF16))
    assert backend.aligns == [128, 256] and backend.graphs == 2


@pytest.mark.parametrize("act,H,I", [("swiglu", 256, 320), ("gelu", 768, 3072), ("swiglu", 1024, 2048)])
@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("least,most", [(4, 20), (30, 60), (200, 400), (900, 2000), (1500, 3000), (20000, 40000)])
def test_a_bounded_row_count_compiles_one_graph(act, H, I, grad, least, most):
    """A token count that the caller says may be anything between two bounds: no rule narrows it, which would have the graph refused
    (ConstraintViolationError). The height is that of the bounds' geometric mean."""
    moe, backend = _layer(act, H, I), _Backend()
    x = torch.randn((least + most) // 2, H, dtype=BF16)
    torch._dynamo.reset()
    torch._dynamo.mark_dynamic(x, 0, min=least, max=most)
    compiled = torch.compile(lambda x: moe(x)[0], fullgraph=True, backend=backend)
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError, match="runs on the GPU only"):
        compiled(x)
    rows = math.isqrt(2 * least * 2 * most)
    assert backend.graphs == 1 and backend.aligns == [scattermoe.choose_align(rows, E, BF16, not grad, (H, I, act == "swiglu"))]


@pytest.mark.parametrize("dtype,rows,grad,height", [
    (torch.float32, 40, False, 128), (torch.float32, 192, True, 128), (torch.float32, 512, False, 256), (BF16, 40, False, 128),
    (BF16, 192, False, 128), (BF16, 40, True, 128), (BF16, 512, True, 256),
])
def test_the_reference_interface(monkeypatch, dtype, rows, grad, height):
    """scattered_experts and an Experts module, eager and traced, at 8 experts of 256 x 320."""
    experts, R = ck.Experts(E, 256, 320, False, 0.02).to(dtype), rows * E
    x = torch.randn(R, 256, dtype=dtype, requires_grad=grad)
    se, ss = torch.arange(E).repeat_interleave(rows), torch.arange(R)
    off = torch.full((E,), rows).cumsum(0)
    seen = []

    def segments(*args):
        seen.append(args[3])
        raise _Stop

    call = lambda x: experts(x, 1, se, ss, off, grouped_in=True, grouped_out=True)
    backend = _Backend()
    _traced(call, x, backend, grad, dynamic=False)
    assert backend.aligns == [height]
    monkeypatch.setattr(scattermoe, "segments_from_sorted", segments)
    monkeypatch.setattr(scattermoe._C, "require_gpu", lambda *t: None)
    with torch.set_grad_enabled(grad), pytest.raises(_Stop):
        call(x)
    assert seen == [height]


def test_graphs_saved_without_a_height_still_call():
    """The operators of the reference's interface took no `align` argument once."""
    for op in (torch.ops.ck_mi355.scattered_experts, torch.ops.ck_mi355.scattered_experts_backward):
        last = op.default._schema.arguments[-1]
        assert last.name == "align" and last.default_value == 0
    meta = lambda *s, dtype=BF16: torch.empty(*s, dtype=dtype, device="meta")
    idx = lambda n: meta(n, dtype=torch.int64)
    out, _ = torch.ops.ck_mi355.scattered_experts(meta(6, 16), meta(4, 8, 16), None, None, idx(12), idx(12), idx(4), 2, False, False)
    assert out.shape == (12, 8)


@pytest.mark.parametrize("experts,H,I,gated,rows,height", [(32, 3456, 896, True, 94, 256), (8, 1152, 8896, True, 136, 256), (8, 1792, 7936, True, 40, 256),
                                                           (16, 1920, 5632, False, 102, 128), (8, 3584, 832, True, 81, 128), (8, 896, 4672, False, 74, 128)])
def test_inference_layers_at_uneven_loads(experts, H, I, gated, rows, height):
    """Heights measured at Zipf(0) to Zipf(1.0) loads: the other one is 5 to 35 % slower."""
    assert scattermoe.choose_align(rows * experts, experts, BF16, True, (H, I, gated)) == height


@pytest.mark.parametrize("experts,H,I,gated,rows,height", [
    (8, 1664, 1088, False, 392, 128), (8, 1408, 3552, True, 168, 128), (8, 1792, 2272, True, 188, 128), (8, 2304, 1440, False, 315, 128),
    (128, 1536, 672, True, 64, 128), (128, 2048, 1408, True, 60, 256), (128, 1024, 2592, True, 140, 256), (64, 3840, 832, True, 120, 256),
])
def test_inference_layers_of_odd_widths_and_many_experts(experts, H, I, gated, rows, height):
    """Measured at Zipf(0), (0.8) and (1.0) loads: the other height is 4 to 41 % slower at each of them (10 to 35 % in the first four,
    whose 128-row launches give few CUs a second tile, or run c_proj on the general kernel)."""
    assert scattermoe.choose_align(rows * experts, experts, BF16, True, (H, I, gated)) == height


@pytest.mark.parametrize("experts", [1, 2, 8, 60, 128, 512])
def test_tiles_of_an_uneven_load(experts):
    """The closed form against the experts' loads one by one: within 10 %, and the tile that one expert's rounding is worth."""
    weights = [(e + 1) ** -0.8 for e in range(experts)]
    assert abs(scattermoe._zipf_sum(experts) / sum(weights) - 1) < 0.006
    for tiles in (0.1, 0.5, 1.3, 3.0, 10.0):  # per expert, on average
        share = tiles * experts / sum(weights)
        want = sum(max(1, math.ceil(share * w)) for w in weights)
        assert abs(scattermoe._zipf_tiles(share, experts) - want) <= 0.1 * want + 1, tiles


@pytest.mark.parametrize("inference", [True, False])
def test_an_unseen_row_count_costs_no_loop_over_the_experts(inference):
    """Lines of the rule that run for it: a server's row count differs from call to call, so that nothing is looked up."""
    def lines(experts):
        ran = 0

        def trace(frame, event, arg):
            nonlocal ran
            if frame.f_code.co_filename != scattermoe.__file__:
                return None
            ran += event == "line"
            return trace

        scattermoe._layer_tiles_kept.cache_clear()
        before = sys.gettrace()
        sys.settrace(trace)
        try:
            scattermoe.choose_align(200 * experts, experts, BF16, inference, (2048, 1408, True))
        finally:
            sys.settrace(before)
        return ran

    assert lines(128) <= lines(8) + 10 <= 200


@pytest.mark.parametrize("rows,layer,quantised", [(6, 16, 16), (7, 32, 32), (22, 32, 32), (23, 64, 64), (30, 64, 64), (31, 128, 64), (40, 128, 64), (41, 128, 256)])
def test_few_rows_per_expert(rows, layer, quantised):
    """The lines between the small tiles; 8 experts of 1,024 x 1,024 take 128 rows behind them."""
    assert scattermoe.choose_align(rows * E, E, BF16, True, (1024, 1024, True)) == layer
    assert scattermoe.choose_align(rows * E, E, BF16, True) == quantised
