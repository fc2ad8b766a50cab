"""Backward kernels that walk the padded grouped layout: the GELU's gradient and the gradient of the experts' biases."""

import ctypes

import pytest
import torch

import cute_kernels
from cute_kernels import _C

pytestmark = pytest.mark.gpu

# rows per expert: none, one, around a 16-row and a 128-row tile, a whole 256-row tile and one row past it
COUNTS = [0, 1, 15, 16, 17, 127, 128, 129, 0, 256, 257, 700]


def _segments(device, align):
    ids = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(COUNTS)])
    seg = cute_kernels.sort_by_expert(ids.to(device), len(COUNTS), align)
    starts = seg.seg_starts.cpu().tolist()
    valid = torch.zeros(seg.max_rows, dtype=torch.bool)
    for e, c in enumerate(COUNTS):
        valid[starts[e] : starts[e] + c] = True
    return seg, starts, valid


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("align,N", [(16, 8), (128, 1032), (256, 520)])
def test_gelu_tanh_backward_of_valid_rows(device, dtype, align, N):
    """The same bits as the flat kernel's on valid rows; pad rows keep what they held."""
    seg, _, valid = _segments(device, align)
    g = torch.Generator().manual_seed(N)
    pre = (2.5 * torch.randn(seg.max_rows, N, generator=g)).to(device, dtype)
    d_act = torch.randn(seg.max_rows, N, generator=g).to(device, dtype)
    pre[~valid.to(device)] = float("nan")  # what an unwritten row may hold
    want, got = torch.empty_like(pre), torch.full_like(pre, 9.0)
    cs = seg.c_struct()
    _C.check(_C.lib().ck_gelu_tanh_bwd(_C.ptr(pre), _C.ptr(d_act), _C.ptr(want), pre.numel(), _C.dtype_code(dtype), _C.stream()))
    _C.check(_C.lib().ck_gelu_tanh_bwd_grouped(_C.ptr(pre), _C.ptr(d_act), N, ctypes.byref(cs), _C.ptr(got), _C.dtype_code(dtype),
                                               _C.stream()))
    assert torch.equal(got.cpu()[valid], want.cpu()[valid])
    assert torch.all(got.cpu()[~valid] == 9.0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("align,N", [(16, 8), (128, 200), (256, 1536)])
def test_expert_bias_gradient(device, dtype, align, N):
    """Against the sum in 64 bits. One rounding to the type, and 32-bit sums of at most 700 terms over 4 waves of 8 accumulators: at
    most 22 additions in an accumulator and 7 in the rows left over, 7 of a wave's, 4 of the waves', each off by 2^-24 of the
    sum of magnitudes."""
    seg, starts, valid = _segments(device, align)
    g = torch.Generator().manual_seed(N)
    d_y = torch.randn(seg.max_rows, N, generator=g).to(dtype)
    d_y[~valid] = float("nan")
    d_bias = torch.empty(len(COUNTS), N, dtype=dtype, device=device)
    on_gpu, cs = d_y.to(device), seg.c_struct()
    _C.check(_C.lib().ck_expert_bias_grad(_C.ptr(on_gpu), N, ctypes.byref(cs), _C.ptr(d_bias), _C.dtype_code(dtype), _C.stream()))
    step = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-24}[dtype]
    for e, c in enumerate(COUNTS):
        rows = d_y[starts[e] : starts[e] + c].double()
        want, bound = rows.sum(0), rows.abs().sum(0) * 40 * 2.0**-24
        off = (d_bias[e].cpu().double() - want).abs()
        assert torch.all(off <= step * want.abs() + bound + 1e-7), (e, c, float(off.max()))


# whole 16-byte pieces of rows (widths of less and more than the 128 columns of a block), and rows that have none: an odd width, and a
# first row off its 16-byte boundary
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,offset", [(120, 0), (136, 0), (1000, 0), (12, 0), (21, 0), (136, 1)])
def test_expert_bias_gradient_by_pieces_and_by_elements(device, dtype, N, offset):
    seg, starts, valid = _segments(device, 128)
    g = torch.Generator().manual_seed(N)
    d_y = torch.randint(-8, 9, (seg.max_rows, N), generator=g).to(dtype)  # sums below 2 ** 13: exact in 32 bits
    d_y[~valid] = float("nan")
    on_gpu, cs = torch.empty(d_y.numel() + offset, dtype=dtype, device=device)[offset:], seg.c_struct()
    on_gpu.copy_(d_y.flatten())
    d_bias = torch.empty(len(COUNTS), N, dtype=dtype, device=device)
    _C.check(_C.lib().ck_expert_bias_grad(_C.ptr(on_gpu), N, ctypes.byref(cs), _C.ptr(d_bias), _C.dtype_code(dtype), _C.stream()))
    for e, c in enumerate(COUNTS):
        assert torch.equal(d_bias[e].cpu(), d_y[starts[e] : starts[e] + c].double().sum(0).to(dtype)), e


# which of the two kernels sums goes by the rows per expert, 350 on average (192 of 32 bits or of many sums): both sides, one expert with none and one with
# nearly all rows
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("total", [3 * 64, 3 * 150, 3 * 250, 3 * 340, 3 * 351, 3 * 700])
@pytest.mark.parametrize("N", [8, 136, 1000])
def test_expert_bias_gradient_of_few_and_many_rows(device, dtype, total, N):
    counts = [5, 0, total - 5]
    seg = cute_kernels.sort_by_expert(torch.tensor([0] * 5 + [2] * (total - 5), dtype=torch.int32, device=device), 3, 128)
    g = torch.Generator().manual_seed(N + total)
    d_y = torch.full((seg.max_rows, N), float("nan"))
    starts, want = seg.seg_starts.cpu().tolist(), torch.zeros(3, N, dtype=torch.float64)
    for e, c in enumerate(counts):
        rows = torch.randint(-8, 9, (c, N), generator=g).float()  # sums below 2 ** 15: exact in 32 bits
        d_y[starts[e] : starts[e] + c], want[e] = rows, rows.double().sum(0)
    on_gpu, cs = d_y.to(dtype).to(device), seg.c_struct()
    d_bias = torch.empty(3, N, dtype=dtype, device=device)
    _C.check(_C.lib().ck_expert_bias_grad(_C.ptr(on_gpu), N, ctypes.byref(cs), _C.ptr(d_bias), _C.dtype_code(dtype), _C.stream()))
    assert torch.equal(d_bias.cpu(), want.to(dtype))
