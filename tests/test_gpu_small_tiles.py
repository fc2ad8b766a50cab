"""GPU parity of the small-row grouped GEMMs (16-, 32- and 64-row tiles: inference batches with few rows per expert), through
the C ABI, against fp32 products of the same operands."""

import pytest
import torch
import torch.nn.functional as F

import cute_kernels
from cute_kernels import _C, fp8, scattermoe
from cute_kernels.modules import moe as moe_module
from oracle import moe_oracle as mo

pytestmark = pytest.mark.gpu

# outputs are fp32 sums rounded once to 16 bits: half a step of bf16 is 2^-9 of the value; 1e-2 as in the other GEMM tests
RTOL = ATOL = 1e-2


def _case(device, T, k, E, align, seed):
    g = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, E, (T * k,), generator=g, dtype=torch.int32)
    ids[ids == 1] = 0  # one empty expert, one with more rows than a tile
    seg = cute_kernels.sort_by_expert(ids.to(device), E, align)
    return g, seg


def _rows(seg):
    """(padded row, expert, flat slot) of every valid row."""
    starts, counts, slot = seg.seg_starts.cpu(), seg.counts.cpu().to(torch.int64), seg.row_slot.cpu()
    return [(p, e, int(slot[p])) for e in range(seg.num_experts) for p in range(int(starts[e]), int(starts[e]) + int(counts[e]))]


# T: a single row, less than a tile, several ragged tiles. K: one step of one wave, a partial step only, an uneven split of
# the steps over the waves with a partial step behind it. N: less than a column tile, ragged, several tiles.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("align", [16, 32, 64])
@pytest.mark.parametrize("T,K,N", [(1, 64, 80), (9, 8, 144), (60, 200, 128), (150, 648, 272)])
@pytest.mark.parametrize("epilogue", ["grouped_bias", "scatter", "swiglu", "swiglu_no_pre", "glu", "gelu"])
def test_small_tiles_match_fp32(device, dtype, align, T, K, N, epilogue):
    k, E = 2, 5
    g, seg = _case(device, T, k, E, align, seed=T + K)
    x = torch.randn(T, K, generator=g).to(dtype)
    w = (0.1 * torch.randn(E, N, K, generator=g)).to(dtype)
    bias = torch.randn(E, N, generator=g).to(dtype)
    rows = _rows(seg)
    want = torch.stack([F.linear(x[s // k].float(), w[e].float()) for _, e, s in rows])
    experts = torch.tensor([e for _, e, _ in rows])
    padded = torch.tensor([p for p, _, _ in rows])
    xd, wd = x.to(device), w.to(device)
    nan = lambda *shape: torch.full(shape, float("nan"), dtype=dtype, device=device)  # noqa: E731
    if epilogue == "scatter":  # grouped input, (token, slot) output
        a = nan(seg.max_rows, K)
        a[padded.to(device)] = torch.stack([x[s // k] for _, _, s in rows]).to(device)
        y = nan(T * k, N)
        scattermoe._gemm(a, 0, wd, seg, _C.CK_EPI_SCATTER, y)
        torch.testing.assert_close(y.cpu().float()[[s for _, _, s in rows]], want, rtol=RTOL, atol=ATOL)
    elif epilogue == "grouped_bias":
        y = nan(seg.max_rows, N)
        scattermoe._gemm(xd, k, wd, seg, _C.CK_EPI_GROUPED, y, aux_in=bias.to(device))
        torch.testing.assert_close(y.cpu().float()[padded], want + bias.float()[experts], rtol=RTOL, atol=ATOL)
        assert torch.isnan(y).sum() == N * (seg.max_rows - len(rows))  # pad rows are left alone
    elif epilogue == "gelu":
        act = nan(seg.max_rows, N)
        scattermoe._gemm(xd, k, wd, seg, _C.CK_EPI_GELU_TANH, None, aux=act)
        torch.testing.assert_close(act.cpu().float()[padded], F.gelu(want.to(dtype).float(), approximate="tanh"), rtol=RTOL, atol=ATOL)
    else:
        act = nan(seg.max_rows, N // 2)
        pre = None if epilogue == "swiglu_no_pre" else nan(seg.max_rows, N)
        scattermoe._gemm(xd, k, wd, seg, _C.CK_EPI_GLU if epilogue == "glu" else _C.CK_EPI_SWIGLU, pre, aux=act)
        fn = (lambda t: F.glu(t, dim=-1)) if epilogue == "glu" else mo.swiglu_packed_torch
        torch.testing.assert_close(act.cpu().float()[padded], fn(want), rtol=2 * RTOL, atol=ATOL)  # two rounded factors
        if pre is not None:
            torch.testing.assert_close(pre.cpu().float()[padded], want, rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("align", [16, 32, 64])
@pytest.mark.parametrize("T,K,N", [(1, 128, 80), (40, 640, 272), (150, 1152, 128)])
def test_small_tiles_fp8(device, align, T, K, N):
    """The same products on e4m3 operands: against the de-quantised fp32 product (exact products, fp32 sums, one rounding)."""
    k, E, dtype = 2, 5, torch.bfloat16
    g, seg = _case(device, T, k, E, align, seed=T + K)
    x8, xs = cute_kernels.quantize_rows_e4m3(torch.randn(T, K, generator=g).to(dtype).to(device))
    w8, ws = cute_kernels.quantize_expert_weights_e4m3((0.1 * torch.randn(E, N, K, generator=g)).to(dtype).to(device))
    xd, wd = x8.cpu().float() * xs.cpu()[:, None], w8.cpu().float() * ws.cpu()[:, :, None]
    rows = _rows(seg)
    want = torch.stack([F.linear(xd[s // k], wd[e]) for _, e, s in rows])
    padded = torch.tensor([p for p, _, _ in rows])
    act = torch.full((seg.max_rows, N // 2), float("nan"), dtype=dtype, device=device)
    fp8._gemm_fp8(x8, xs, k, w8, ws, seg, _C.CK_EPI_SWIGLU, None, act, dtype)
    torch.testing.assert_close(act.cpu().float()[padded], mo.swiglu_packed_torch(want), rtol=2 * RTOL, atol=ATOL)
    a8 = torch.zeros(seg.max_rows, K, dtype=torch.uint8, device=device)
    scale = torch.ones(seg.max_rows, device=device)
    at = padded.to(device)
    src = torch.tensor([s // k for _, _, s in rows], device=device)
    a8[at], scale[at] = x8.view(torch.uint8)[src], xs[src]
    y = torch.full((T * k, N), float("nan"), dtype=dtype, device=device)
    fp8._gemm_fp8(a8.view(torch.float8_e4m3fn), scale, 0, w8, ws, seg, _C.CK_EPI_SCATTER, y, None, dtype)
    torch.testing.assert_close(y.cpu().float()[[s for _, _, s in rows]], want, rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("rows", [31, 100, 101, 300])
def test_inference_on_128_row_tiles_matches_a_forward_on_256(device, monkeypatch, gated, rows):
    """Narrow layers between the small tiles and 512 rows per expert: the same sums as on 256-row tiles with what a backward
    pass needs kept, in another order at most."""
    E, H, I = 8, 256, 320
    assert scattermoe.choose_align(rows * E, E, torch.bfloat16, True, (H, I, gated)) == 128
    torch.manual_seed(rows)
    act = cute_kernels.swiglu_packed_cute if gated else torch.nn.GELU(approximate="tanh")
    moe = cute_kernels.MoE(E, 2, H, I, act, gated, not gated, 0.05).to(device, torch.bfloat16)
    x = torch.randn(rows * E // 2, H, device=device).to(torch.bfloat16)
    with torch.no_grad():
        got, _ = moe(x)
    monkeypatch.setattr(moe_module, "choose_align", lambda *args: 256)
    want, _ = moe(x)
    torch.testing.assert_close(got.float(), want.detach().float(), rtol=RTOL, atol=ATOL)


# weights on 128-byte boundaries throughout, with another row pitch, and with another first row; one line a row, several, and a part of
# one. Column tiles of 64 (32 outputs with a gate) and a rest; with 4,104 columns, 520 to 715 tiles: whole rounds of chunks over the
# XCDs and a rest, at every height, with experts of several row tiles
@pytest.mark.parametrize("align", [16, 32, 64])
@pytest.mark.parametrize("K,offset", [(64, 0), (320, 0), (328, 0), (320, 8), (32, 0)])
@pytest.mark.parametrize("columns", [8, 200, 1032, 4104])
def test_weight_lines(device, align, K, offset, columns):
    g = torch.Generator().manual_seed(K + columns)
    counts = [0, 2 * align + 3, 1, 0, align, 5, 70, 0]
    ids = torch.arange(len(counts), dtype=torch.int32).repeat_interleave(torch.tensor(counts)).to(device)
    seg = scattermoe.sort_by_expert(ids, len(counts), align)
    a = torch.full((seg.max_rows, K), float("nan"), dtype=torch.bfloat16)
    rows = [torch.randint(-2, 3, (c, K), generator=g).to(torch.bfloat16) for c in counts]
    starts = seg.seg_starts.cpu().tolist()
    for e, c in enumerate(counts):
        a[starts[e] : starts[e] + c] = rows[e]
    w = torch.randint(-1, 2, (len(counts), columns, K), generator=g).to(torch.bfloat16)
    wd = torch.empty(w.numel() + offset, dtype=torch.bfloat16, device=device)[offset:].view(w.shape).copy_(w)
    y = torch.full((seg.max_rows, columns), 1000.0, dtype=torch.bfloat16, device=device)
    scattermoe._gemm(a.to(device), 0, wd, seg, _C.CK_EPI_GROUPED, y)
    y = y.cpu().float()
    for e, c in enumerate(counts):
        want = (rows[e].float() @ w[e].float().t()).to(torch.bfloat16).float()  # whole numbers, exact in fp32 and rounded once
        assert torch.equal(y[starts[e] : starts[e] + c], want), e


# Four experts have rows, of 16 to 64 a tile: 128 column tiles of 64 (the last one ragged) and so on, that is a launch that goes out in
# halves of tiles, one of more than half a round, whole rounds, and these behind a whole round
@pytest.mark.parametrize("align", [16, 32, 64])
@pytest.mark.parametrize("N", [2032, 2064, 4096, 4112, 6160])
@pytest.mark.parametrize("epilogue", ["grouped_bias", "scatter", "swiglu", "fp8"])
def test_last_round_in_halves(device, align, N, epilogue):
    if epilogue == "fp8":
        test_small_tiles_fp8(device, align, 9, 1152, N)
    else:
        test_small_tiles_match_fp32(device, torch.bfloat16, align, 9, 200, N, epilogue)
