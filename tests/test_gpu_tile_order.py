"""The order in which the workgroups of a grouped GEMM take its tiles: every tile of every expert once, whatever its number
of row tiles (none, one, a whole group, one more than a group) and whichever split over the XCDs the grid gets."""

import pytest
import torch

from cute_kernels import _C, scattermoe

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _segments(counts, align=256):
    ids = torch.arange(len(counts), dtype=torch.int32).repeat_interleave(torch.tensor(counts)).to(DEV)
    return scattermoe.sort_by_expert(ids, len(counts), align)


def _operand(seg, width, counts, g):
    """Padded grouped rows with small whole numbers, so that products and sums are exact; and the rows of every expert."""
    a = torch.full((seg.max_rows, width), float("nan"), dtype=torch.bfloat16)
    starts = seg.seg_starts.cpu().tolist()
    for e, c in enumerate(counts):
        a[starts[e] : starts[e] + c] = torch.randint(-2, 3, (c, width), generator=g).to(torch.bfloat16)
    return a.to(DEV), [a[starts[e] : starts[e] + c].float() for e, c in enumerate(counts)]


@pytest.mark.parametrize("columns", [264, 2816])  # 2 and 11 column tiles
@pytest.mark.parametrize("counts", [[2300, 0, 1, 256, 257, 2049], [0, 0, 5], [300] * 9])
def test_forward_tiles(counts, columns):
    g = torch.Generator().manual_seed(0)
    seg = _segments(counts)
    a, rows = _operand(seg, 64, counts, g)
    w = torch.randint(-2, 3, (len(counts), columns, 64), generator=g).to(torch.bfloat16)
    y = torch.full((seg.max_rows, columns), 1000.0, dtype=torch.bfloat16, device=DEV)
    scattermoe._gemm(a, 0, w.to(DEV), seg, _C.CK_EPI_GROUPED, y)
    y = y.cpu().float()
    for e, c in enumerate(counts):
        first = int(seg.seg_starts[e])
        assert torch.equal(y[first : first + c], rows[e] @ w[e].float().t())  # |sum| <= 256: exact in bf16


# the general kernel: fewer than two row tiles per expert (groups over all of them, one of 20 included), exactly two, and more
@pytest.mark.parametrize("align,K", [(128, 64), (128, 40), (256, 40)])
@pytest.mark.parametrize("tiles", [[1, 0, 1, 1], [3, 0, 1, 3], [4, 0, 2, 2], [1] * 20, [2] * 9, [0, 0, 0, 9]])
def test_forward_tiles_of_the_general_kernel(tiles, align, K):
    g = torch.Generator().manual_seed(1)
    counts = [max(0, t * align - 3 * e) for e, t in enumerate(tiles)]
    seg = _segments(counts, align)
    a, rows = _operand(seg, K, counts, g)
    w = torch.randint(-2, 3, (len(counts), 648, K), generator=g).to(torch.bfloat16)
    y = torch.full((seg.max_rows, 648), 1000.0, dtype=torch.bfloat16, device=DEV)
    scattermoe._gemm(a, 0, w.to(DEV), seg, _C.CK_EPI_GROUPED, y)
    y = y.cpu().float()
    for e, c in enumerate(counts):
        first = int(seg.seg_starts[e])
        assert torch.equal(y[first : first + c], rows[e] @ w[e].float().t())


# 256 x 256 tiles: 32 x 1 (4 per XCD, an eighth of a round of chunks: slices), 32 x 8 (one round: slices, or chunks of 32 from 4,096
# rows per expert on), 16 x 1 (chunks of 16, or slices from 2,048 rows on), 16 x 8 (one round: chunks of 16), 11 x 2 (chunks of 16;
# 8 experts: 176 tiles, whole rounds of chunks and a rest), 1 x 1; the longer side is the rows' or the columns'.
# The first three lists average fewer than 512 rows: 128 x 256 tiles, in slices of 8 of them or chunks of 32, contractions of one
# step of 32 rows, of two and more, ragged and whole; ragged tiles of both kernels.
@pytest.mark.parametrize("M,N", [(8192, 256), (8192, 2048), (256, 4096), (4096, 2048), (2816, 512), (512, 2568), (256, 256), (328, 264)])
@pytest.mark.parametrize(
    "counts",
    [[70, 0, 64, 65, 1, 128, 3, 200], [33], [31, 32, 97, 511], [600, 0, 1100, 513, 512, 700, 3, 1500], [4000, 4200, 0, 8300]],
)
def test_weight_gradient_tiles(counts, M, N):
    g = torch.Generator().manual_seed(1)
    seg = _segments(counts)
    a, a_rows = _operand(seg, M, counts, g)
    b, b_rows = _operand(seg, N, counts, g)
    dw = torch.full((len(counts), M, N), 1000.0, dtype=torch.bfloat16, device=DEV)
    scattermoe._gemm_dw_rows(a, b, seg, dw)
    for e in range(len(counts)):
        # sums below 2^24: exact in fp32, one rounding
        expect = (a_rows[e].to(DEV).t().contiguous() @ b_rows[e].to(DEV)).to(torch.bfloat16)
        assert torch.equal(dw[e], expect), e


# 6 experts, 13 row tiles x 20 / 25 / 28 column tiles: a last round of 4 / 69 / 108 tiles, in 4 / 3 / 2 parts where that takes 40 of
# its K steps off: 54, 60, 80 steps are the fewest, 53 too few for any
@pytest.mark.parametrize("columns,K", [(5120, 54 * 64), (6400, 60 * 64), (7168, 80 * 64), (5120, 53 * 64)])
@pytest.mark.parametrize("weights", ["as columns x contraction", "as stored by their owner"])
def test_split_last_round(monkeypatch, weights, columns, K):
    """The same launch split and unsplit: equal up to the fp32 re-association of a few partial sums, bit for bit from one split
    launch to the next, and bit for bit to the unsplit one where the rule says no."""
    counts = [700, 513, 600, 0, 512, 400]
    seg = _segments(counts)
    tiles = sum(-(-c // 256) for c in counts) * (columns // 256)
    assert 0 < tiles % 256 <= 128
    g = torch.Generator(device=DEV).manual_seed(2)
    a = torch.randn(seg.max_rows, K, generator=g, device=DEV).to(torch.bfloat16)
    shape = (len(counts), columns, K) if weights == "as columns x contraction" else (len(counts), K, columns)
    w = (torch.randn(shape, generator=g, device=DEV) * K**-0.5).to(torch.bfloat16)
    outs = []
    for split in (True, True, False):
        monkeypatch.setattr(scattermoe.options, "gemm_split", split)
        out = torch.zeros(seg.max_rows, columns, dtype=torch.bfloat16, device=DEV)
        if weights == "as columns x contraction":
            scattermoe._gemm(a, 0, w, seg, _C.CK_EPI_GROUPED, out)
        else:
            scattermoe._gemm_dx(a, w, seg, _C.CK_EPI_GROUPED, out)
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    same = (outs[0] == outs[2]).float().mean()
    if K == 53 * 64:
        assert same == 1
    else:  # a last round of 4 of 260 tiles and more: some element of its tiles rounds the other way
        assert 0.99 < float(same) < 1
        # 256 k of K terms ~ N(0, 1 / K): sums differ by a few 2 ** -24, one rounding step of bf16 (2 ** -8) where they straddle
        torch.testing.assert_close(outs[0].float(), outs[2].float(), rtol=2.0**-7, atol=2.0**-16)


# 13 row tiles x 20 / 28 column tiles: a last round of 4 / 108 tiles, in 4 / 2 parts, or whole (53 steps)
@pytest.mark.parametrize("columns,K", [(5120, 54 * 64), (7168, 80 * 64), (5120, 53 * 64)])
@pytest.mark.parametrize("epilogue,bias", [("swiglu", False), ("gelu", True), ("gelu", False), ("scatter", True)])
def test_split_last_round_of_the_activation_and_bias_epilogues(monkeypatch, epilogue, bias, columns, K):
    counts = [700, 513, 600, 0, 512, 400]
    seg = _segments(counts)
    g = torch.Generator(device=DEV).manual_seed(3)
    a = torch.randn(seg.max_rows, K, generator=g, device=DEV).to(torch.bfloat16)
    gate = 2 if epilogue == "swiglu" else 1
    w = (torch.randn((len(counts), columns, K), generator=g, device=DEV) * K**-0.5).to(torch.bfloat16)
    bias = torch.randn(len(counts), columns, generator=g, device=DEV).to(torch.bfloat16) if bias else None
    code = {"swiglu": _C.CK_EPI_SWIGLU, "gelu": _C.CK_EPI_GELU_TANH, "scatter": _C.CK_EPI_SCATTER}[epilogue]
    outs = []
    for split in (True, True, False):
        monkeypatch.setattr(scattermoe.options, "gemm_split", split)
        y = torch.zeros(sum(counts) if epilogue == "scatter" else seg.max_rows, columns, dtype=torch.bfloat16, device=DEV)
        aux = None if epilogue == "scatter" else torch.zeros(seg.max_rows, columns // gate, dtype=torch.bfloat16, device=DEV)
        scattermoe._gemm(a, 0, w, seg, code, y, aux=aux, aux_in=bias)
        outs.append(torch.cat([t.flatten() for t in (y, aux) if t is not None]))
    assert torch.equal(outs[0], outs[1])
    differ = int((outs[0] != outs[2]).sum())
    if K == 53 * 64:
        assert differ == 0
    else:
        assert 0 < differ < 0.01 * outs[0].numel()
        # sums of K terms ~ N(0, 1 / K) differ by a few 2 ** -24; a pre-activation may then round to the next bf16 value (2 ** -8
        # of it), and so may the output. Gate: x silu'(x) / silu(x) is at most 1 + |x|, |x| < 6: 7 + 2 steps of 2 ** -8 at most.
        # GELU: |x gelu'(x)| < 0.2 for negative x, 0.2 * 2 ** -8 in all, and at most 1.2 steps of the output for positive ones.
        torch.testing.assert_close(outs[0].float(), outs[2].float(), rtol=2.0**-4.8, atol=2.0**-10)
