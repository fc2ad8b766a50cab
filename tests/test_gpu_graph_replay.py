"""Captured HIP graphs: a replay computes from the inputs it finds, whatever earlier replays and eager calls left behind."""

import pytest
import torch

import cute_kernels
from cute_kernels import _C, scattermoe

pytestmark = pytest.mark.gpu


def _splits(seg, experts, columns, K):
    """Whether a launch on 256-row tiles splits its last round: at most half full, and 40 K steps or more saved by its parts."""
    tail, steps = int(seg.seg_starts[experts]) // 256 * -(-columns // 256) % 256, K // 64
    return 0 < tail <= 128 and steps - -(-steps // min(4, 256 // tail)) >= 40


@pytest.mark.parametrize("tokens,hidden,inter", [(300, 1024, 3456), (520, 2048, 3840)])
def test_replays_of_a_layer_with_a_split_last_round(device, tokens, hidden, inter):
    """A layer whose c_proj GEMM is the graph's only launch that splits its last round of tiles, on a stream that runs nothing
    else: every replay finds the workspace as the replay before left it. Each one equals the eager layer bit for bit (the
    same kernels on the same layout; the parts of a split tile are added in a fixed order)."""
    E, k = 4, 2
    g = torch.Generator(device=device).manual_seed(7)
    rand = lambda *shape: torch.randn(*shape, device=device, generator=g)
    w_fc, w_proj = (0.03 * rand(E, 2 * inter, hidden)).bfloat16(), (0.03 * rand(E, hidden, inter)).bfloat16()
    ids = torch.stack([torch.randperm(E, device=device, generator=g)[:k] for _ in range(tokens)]).int()
    x, gates = rand(tokens, hidden).bfloat16(), torch.rand(tokens, k, device=device, generator=g).bfloat16()

    def layer():
        return scattermoe.swiglu_experts(x, w_fc, w_proj, gates, cute_kernels.sort_by_expert(ids, E, 256))

    with torch.no_grad():
        seg = cute_kernels.sort_by_expert(ids, E, 256)
        assert _splits(seg, E, hidden, inter)  # the c_proj launch
        layer()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=torch.cuda.Stream(device)):
            out = layer()
        for _ in range(4):
            x.copy_(rand(tokens, hidden))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, layer())


@pytest.mark.parametrize("steps", [53, 54])
@pytest.mark.parametrize("form", ["forward", "input gradient"])
def test_a_graph_holds_a_workspace_only_where_a_launch_can_split(device, form, steps):
    """53 K steps: no share of a tile's contraction is 40 steps shorter than the whole, whatever the number of tiles."""
    E, N, K = 4, 512, 64 * steps
    ids = torch.randint(0, E, (600,), device=device, dtype=torch.int32)
    seg = cute_kernels.sort_by_expert(ids, E, 256)
    a, out = (torch.zeros(seg.max_rows, n, device=device, dtype=torch.bfloat16) for n in (K, N))
    w = torch.zeros(E, *((N, K) if form == "forward" else (K, N)), device=device, dtype=torch.bfloat16)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        if form == "forward":
            scattermoe._gemm(a, 0, w, seg, _C.CK_EPI_GROUPED, out)
        else:
            scattermoe._gemm_dx(a, w, seg, _C.CK_EPI_GROUPED, out)
    taken = torch.cuda.max_memory_allocated() - before
    assert (taken >= _C.lib().ck_grouped_gemm_workspace_bytes()) == (steps == 54)  # a capture takes a little for itself


def test_graphs_that_count_do_not_depend_on_each_other(device):
    """Two graphs captured on one stream, in memory that earlier replays have used: the second one replayed first, then either,
    with eager calls on the capture stream in between."""
    stream = torch.cuda.Stream(device)
    ids = torch.randint(0, 60, (50000,), device=device, dtype=torch.int32)
    want = torch.bincount(ids, minlength=60)
    dirty = torch.cuda.CUDAGraph()
    with torch.cuda.graph(dirty, stream=stream):
        used = [torch.full((1 << 18,), 7, dtype=torch.int32, device=device) for _ in range(4)]
    dirty.replay()
    torch.cuda.synchronize()
    del used
    graphs = []
    for _ in range(2):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, pool=dirty.pool()):
            out = cute_kernels.continuous_count_cute(ids, 60)
        graphs.append((graph, out))
    for i in (1, 0, 1, 1, 0):
        graph, out = graphs[i]
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.long(), want), i
        with torch.cuda.stream(stream):
            eager = cute_kernels.continuous_count_cute(ids, 60)
        torch.cuda.synchronize()
        assert torch.equal(eager.long(), want)


@pytest.mark.parametrize("act", ["swiglu", "gelu"])
@pytest.mark.parametrize("tokens,inter", [(40, 1024), (700, 3456)])  # tiles of 128 rows; of 256 rows with split last rounds
def test_replays_of_a_training_step_of_the_experts(device, act, tokens, inter):
    """Forward and backward of the expert block in one graph (the backward launches from the autograd engine's thread), replayed
    on other inputs with eager steps in between: outputs and gradients bit for bit those of an eager step."""
    E, k, hidden = 4, 2, 1024
    g = torch.Generator(device=device).manual_seed(3)
    rand = lambda *shape: torch.randn(*shape, device=device, generator=g)
    w_fc = (0.03 * rand(E, 2 * inter if act == "swiglu" else inter, hidden)).bfloat16().requires_grad_()
    w_proj = (0.03 * rand(E, hidden, inter)).bfloat16().requires_grad_()
    ids = torch.stack([torch.randperm(E, device=device, generator=g)[:k] for _ in range(tokens)]).int()
    x, dy = rand(tokens, hidden).bfloat16().requires_grad_(), rand(tokens, hidden).bfloat16()
    gates = torch.rand(tokens, k, device=device, generator=g).bfloat16().requires_grad_()
    leaves = (x, gates, w_fc, w_proj)
    align = 128 if tokens < 100 else 256
    if align == 256:  # c_proj, and d_x through c_fc's weights
        assert _splits(cute_kernels.sort_by_expert(ids, E, align), E, hidden, inter)

    def step():
        seg = cute_kernels.sort_by_expert(ids, E, align)
        if act == "swiglu":
            y = scattermoe.swiglu_experts(x, w_fc, w_proj, gates, seg)
        else:
            y = scattermoe.experts_up(x, w_fc, seg, k, gelu_tanh=True, down=(w_proj, gates, None))
        return [y.detach(), *torch.autograd.grad(y, leaves, dy)]

    warm = torch.cuda.Stream(device)
    warm.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(warm):
        step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for _ in range(4):
        with torch.no_grad():
            x.copy_(rand(tokens, hidden))
            dy.copy_(rand(tokens, hidden))
            w_fc.mul_(0.99)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, step()):
            assert torch.equal(a, b)
