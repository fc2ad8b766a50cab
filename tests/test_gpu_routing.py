"""GPU parity (through the C ABI) for the integer stages: histogram/offsets, top-k routing, stable sort by expert.
Bit-exact against oracle/ck_oracle.c and against the committed fixtures."""

import os

import numpy as np
import pytest
import torch

import cute_kernels
from cute_kernels import _C
from oracle import integer_oracle as io

pytestmark = pytest.mark.gpu

GOLDEN = np.load(os.path.join(os.path.dirname(__file__), "golden", "routing_fixtures.npz"))


def _count_sizes():
    sizes = set()
    for i in range(15):  # the reference's 1-D size grid (tests/test_commons.py:30-40), thinned on j
        for j in (0, 1, 3, 7, 9):
            sizes.add(2**i + j)
    rng = np.random.default_rng(0)
    sizes.update(int(v) for v in rng.integers(2000, 4000, size=6))
    return sorted(sizes)


@pytest.mark.parametrize("dtype", [torch.int32, torch.long])
def test_continuous_count_reference_grid(device, dtype):
    # continuous_count_test.py:19-41 of the reference: ids ~ randint(0, 72), exact match with bincount
    g = torch.Generator().manual_seed(42)
    for n in _count_sizes():
        x = torch.randint(0, 72, (n,), generator=g, dtype=dtype)
        got = cute_kernels.continuous_count_cute(x.to(device), 72)
        assert got.dtype == torch.uint32 and got.shape == (72,)
        np.testing.assert_array_equal(got.cpu().numpy(), io.count(x.numpy(), 72), err_msg=f"n={n}")


@pytest.mark.parametrize("bins", [2, 8, 9, 16, 17, 64, 1000, 1024, 1025, 16384])
@pytest.mark.parametrize("dtype", [torch.int32, torch.long])
def test_count_offsets_bin_ranges(device, bins, dtype):
    g = torch.Generator().manual_seed(bins)
    for n in (0, 5, 70001, 1 << 20):
        x = torch.randint(0, bins, (n,), generator=g, dtype=dtype)
        counts, ends, starts = cute_kernels.continuous_count_and_offsets_cute(x.to(device), bins)
        c = io.count(x.numpy(), bins)
        e, s = io.offsets(c)
        np.testing.assert_array_equal(counts.cpu().numpy(), c)
        np.testing.assert_array_equal(ends.cpu().numpy(), e)
        np.testing.assert_array_equal(starts.cpu().numpy(), s)


def test_count_golden_c1_and_repeat_calls(device):
    ids = np.random.default_rng(int(GOLDEN["c1_seed"][0])).integers(0, 64, size=65536, dtype=np.int64)
    x = torch.from_numpy(ids).to(torch.int32).to(device)
    for _ in range(3):  # the workspace must come back to zero after every call
        counts, ends, starts = cute_kernels.continuous_count_and_offsets_cute(x, 64)
        np.testing.assert_array_equal(counts.cpu().numpy(), GOLDEN["c1_counts"])
        np.testing.assert_array_equal(ends.cpu().numpy(), GOLDEN["c1_ends"])
        np.testing.assert_array_equal(starts.cpu().numpy(), GOLDEN["c1_starts"])


def test_count_misaligned_views_out_of_range_and_shortcut(device):
    g = torch.Generator().manual_seed(5)
    base = torch.randint(-3, 80, (100003,), generator=g, dtype=torch.int32)
    for off in (1, 2, 3):
        x = base[off:]
        got = cute_kernels.continuous_count_cute(x.to(device)[0:], 72)  # keep the odd start through a device slice
        xd = base.to(device)[off:]
        got = cute_kernels.continuous_count_cute(xd, 72)
        np.testing.assert_array_equal(got.cpu().numpy(), io.count(x.numpy(), 72))
    out = cute_kernels.continuous_count_cute(torch.zeros(7, 3, device=device), 1)
    assert out.tolist() == [21] and out.dtype == torch.uint32
    strided = torch.arange(0, 64, dtype=torch.long, device=device).repeat(4)[::2]
    np.testing.assert_array_equal(
        cute_kernels.continuous_count_cute(strided, 64).cpu().numpy(), io.count(strided.cpu().numpy(), 64)
    )


# narrow and wide blocks, one trip and several: 1, 16 and 512 blocks of 512 threads (8,192 int32 or 4,096 int64 ids each), 1 and
# 512 of 1,024 threads, and one id more; the most bins with a histogram per wave and the fewest with one for all waves
@pytest.mark.parametrize("dtype", [torch.int32, torch.long])
@pytest.mark.parametrize("bins", [1, 8, 9, 32, 33, 128, 1024, 1025])
def test_count_launch_forms(device, bins, dtype):
    per_block = 8192 if dtype == torch.int32 else 4096
    for n in (1, 512, per_block, per_block + 1, 2 * per_block, 2 * per_block + 1, 16 * per_block, 16 * per_block + 1, 512 * per_block, 512 * per_block + 1, 1024 * per_block + 1):
        x = torch.randint(0, bins, (n,), dtype=dtype, device=device)
        expect = torch.bincount(x, minlength=bins).cpu().numpy()
        for repeat in range(2):  # tickets and accumulators come back to zero
            counts, ends, _ = cute_kernels.continuous_count_and_offsets_cute(x, bins)
            np.testing.assert_array_equal(counts.cpu().numpy(), expect, err_msg=f"n={n} call {repeat}")
            np.testing.assert_array_equal(ends.cpu().numpy(), expect.cumsum())


# one accumulator for all 512 blocks (4,097 to 8,192 bins), two and three, and one without groups of tickets: additions queue up
@pytest.mark.parametrize("bins", [3000, 4097, 5000, 8192, 8193, 16384])
def test_count_many_blocks_on_few_accumulators(device, bins):
    x = torch.randint(0, bins, (512 * 16384 + 1,), dtype=torch.int32, device=device)
    expect = torch.bincount(x, minlength=bins)
    for _ in range(5):
        assert torch.equal(cute_kernels.continuous_count_cute(x, bins).long(), expect)


def test_count_large_sum_property(device):
    # full-size property at 2^28 ids (1 GiB): counts sum to N and match a strided sample's histogram scaled check
    n = 1 << 28
    x = torch.randint(0, 64, (n,), dtype=torch.int32, device=device)
    counts, ends, starts = cute_kernels.continuous_count_and_offsets_cute(x, 64)
    c = counts.cpu().numpy().astype(np.int64)
    assert int(c.sum()) == n and int(ends[-1]) == n and int(starts[0]) == 0
    np.testing.assert_array_equal(c, torch.bincount(x, minlength=64).cpu().numpy())


@pytest.mark.parametrize("T,E,k", [(16384, 64, 2), (1000, 8, 2), (777, 8, 1), (513, 128, 8), (300, 6, 4), (64, 1000, 32), (5, 3, 3), (129, 72, 7)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_route_topk_softmax_matches_oracle(device, T, E, k, dtype):
    g = torch.Generator().manual_seed(42)
    logits = torch.randn(T, E, generator=g).to(dtype)  # bf16 rounding makes ties common (about 3% of C2 rows)
    sel, gates, vals = cute_kernels.route_topk_softmax_raw(logits.to(device), k)
    o_sel, o_gates, o_vals = io.topk_softmax(logits.float().numpy(), k)
    np.testing.assert_array_equal(sel.cpu().numpy(), o_sel)  # bit-exact, ties included (lowest index first)
    np.testing.assert_array_equal(vals.float().cpu().numpy(), o_vals)
    np.testing.assert_allclose(gates.cpu().numpy(), o_gates, rtol=2e-6, atol=1e-7)
    # and against torch.topk where it is defined: the values
    np.testing.assert_array_equal(vals.float().cpu().numpy(), logits.float().topk(k, dim=-1).values.numpy())


# groups of 1, 2, 8, 16 and 64 lanes: as many selections as lanes (a lane writes one each), and one more (lane 0 writes them all)
@pytest.mark.parametrize("E,k", [(8, 1), (8, 2), (16, 2), (16, 3), (64, 8), (64, 9), (128, 16), (128, 17), (512, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_route_selections_and_lanes_of_a_group(device, E, k, dtype):
    logits = torch.randn(333, E, generator=torch.Generator().manual_seed(E + k)).to(dtype)
    sel, gates, vals = cute_kernels.route_topk_softmax_raw(logits.to(device), k)
    o_sel, o_gates, o_vals = io.topk_softmax(logits.float().numpy(), k)
    np.testing.assert_array_equal(sel.cpu().numpy(), o_sel)
    np.testing.assert_array_equal(vals.float().cpu().numpy(), o_vals)
    np.testing.assert_allclose(gates.cpu().numpy(), o_gates, rtol=2e-6, atol=1e-7)
    both, long = (cute_kernels.route_topk_softmax(logits.to(device), k, long_indices=wide) for wide in (False, True))
    assert both[1].dtype == torch.int32 and long[1].dtype == torch.long and torch.equal(both[1].long(), long[1]) and torch.equal(both[1].cpu(), sel.cpu())
    assert torch.equal(both[0].cpu(), gates.cpu().to(both[0].dtype))


def test_route_special_values(device):
    row = torch.tensor([[1.0, 3.0, 3.0, -0.0, 0.0, 3.0, float("nan"), 2.0]])
    sel, _, _ = cute_kernels.route_topk_softmax_raw(row.to(device), 5)
    assert sel.tolist() == [[6, 1, 2, 5, 7]]
    sel, _, _ = cute_kernels.route_topk_softmax_raw(torch.tensor([[0.0, -0.0, -0.0, 0.0]], device=device), 4)
    assert sel.tolist() == [[0, 1, 2, 3]]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("E,k", [(3, 3), (8, 2), (16, 6), (60, 8), (128, 8), (200, 4), (1000, 32), (1024, 9)])
def test_route_16_bit_keys_order_every_value(device, E, k, dtype):
    """16-bit logits are ordered by 32-bit keys of their own, fp32 ones by 64-bit keys: the same selections, values and gates
    for every bit pattern (zeros of both signs, subnormals, infinities, NaNs), ties included."""
    g = torch.Generator().manual_seed(E)
    bits = torch.randint(-(1 << 15), 1 << 15, (331, E), generator=g, dtype=torch.int32).to(torch.int16)
    special = torch.tensor([0, -32768, 1, -32767, 0x7F80, 0x7C00, 0x7FFF, -1], dtype=torch.int16)  # 0, -0, subnormals, inf, NaN
    mask = torch.rand(331, E, generator=g) < torch.linspace(0, 1, 331)[:, None]
    bits = torch.where(mask, special[torch.randint(0, 8, (331, E), generator=g)], bits)
    logits = bits.view(dtype).to(device)
    sel, gates, vals = cute_kernels.route_topk_softmax_raw(logits, k)
    sel32, gates32, vals32 = cute_kernels.route_topk_softmax_raw(logits.float(), k)
    assert torch.equal(sel, sel32)
    torch.testing.assert_close(gates, gates32, rtol=0, atol=0, equal_nan=True)
    torch.testing.assert_close(vals.float(), vals32, rtol=0, atol=0, equal_nan=True)


def test_route_autograd_matches_torch(device):
    g = torch.Generator().manual_seed(1)
    logits = torch.randn(257, 16, generator=g)  # fp32, no ties
    a = logits.clone().to(device).requires_grad_()
    b = logits.clone().requires_grad_()
    gates, sel = cute_kernels.route_topk_softmax(a, 4)
    v, i = b.topk(4, dim=-1)
    ref = torch.softmax(v.float(), dim=-1)
    assert sel.dtype == torch.long and torch.equal(sel.cpu(), i)
    w = torch.randn(257, 4, generator=g)
    (gates * w.to(device)).sum().backward()
    (ref * w).sum().backward()
    torch.testing.assert_close(gates.cpu(), ref, rtol=2e-6, atol=1e-7)
    torch.testing.assert_close(a.grad.cpu(), b.grad, rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_route_backward_takes_the_unrounded_gate_gradient_where_it_arrived_rounded(device, dtype):
    """ck_route_topk_softmax_bwd_exact against ck_route_topk_softmax_bwd fed with the gradient it has to pick: the fp32
    d_gates where the 16-bit gradient that arrived is that value rounded, the arrived value elsewhere (here every third
    row was doubled on its way, as a hook on the gates would). Bit-exact: same kernel arithmetic on the same inputs."""
    from cute_kernels import _C

    T, E, k = 777, 24, 4
    g = torch.Generator().manual_seed(5)
    logits = torch.randn(T, E, generator=g).to(dtype).to(device)
    sel, gates, _ = cute_kernels.route_topk_softmax_raw(logits, k)
    exact = torch.randn(T, k, generator=g).to(device)
    arrived = exact.to(dtype)
    arrived[::3] *= 2
    picked = torch.where(exact.to(dtype) == arrived, exact, arrived.float())
    assert 0 < int((picked != exact).sum()) < T * k
    lib = _C.lib()
    got = torch.full((T, E), 7.0, dtype=dtype, device=device)
    want = torch.full((T, E), 9.0, dtype=dtype, device=device)
    with torch.cuda.device(device):
        _C.check(lib.ck_route_topk_softmax_bwd_exact(_C.ptr(gates), _C.ptr(exact), _C.ptr(arrived), _C.ptr(sel), T, E, k,
                                                     _C.ptr(got), _C.dtype_code(dtype), _C.stream()))
        _C.check(lib.ck_route_topk_softmax_bwd(_C.ptr(gates), _C.ptr(picked), _C.ptr(sel), T, E, k, _C.ptr(want),
                                               _C.dtype_code(dtype), _C.stream()))
    assert torch.equal(got, want)
    # against autograd of softmax over the selected logits with the picked gradient
    v = torch.gather(logits.float(), 1, sel.long()).requires_grad_()
    torch.softmax(v, -1).backward(picked)
    ref = torch.zeros(T, E, device=device).scatter_(1, sel.long(), v.grad)
    torch.testing.assert_close(got.float(), ref, rtol=1e-2, atol=1e-3)
    rc = lib.ck_route_topk_softmax_bwd_exact(_C.ptr(gates), _C.ptr(exact), _C.ptr(exact), _C.ptr(sel), T, E, k, _C.ptr(got),
                                             _C.CK_F32, _C.stream())
    assert rc != 0  # fp32 gradients have nothing to recover


def _check_sort(device, ids: torch.Tensor, E: int, align: int):
    seg = cute_kernels.sort_by_expert(ids.to(device), E, align)
    idn = ids.numpy().astype(np.int64)
    se, ss = io.sort_by_expert(idn, E)
    c = io.count(idn, E)
    e, s = io.offsets(c)
    np.testing.assert_array_equal(seg.sorted_expert_idxs.cpu().numpy(), se)
    np.testing.assert_array_equal(seg.sorted_scattered_idxs.cpu().numpy(), ss)
    np.testing.assert_array_equal(seg.counts.cpu().numpy(), c)
    np.testing.assert_array_equal(seg.ends.cpu().numpy(), e)
    np.testing.assert_array_equal(seg.starts.cpu().numpy(), s)
    o_seg_starts, o_row_slot, o_tile = io.segments(c, ss, align, seg.max_rows)
    np.testing.assert_array_equal(seg.seg_starts.cpu().numpy(), o_seg_starts)
    np.testing.assert_array_equal(seg.tile_expert.cpu().numpy()[: seg.max_rows // align], o_tile)
    got_slot = seg.row_slot.cpu().numpy()[: seg.max_rows]
    valid = o_row_slot >= 0  # pad rows are left unwritten by the kernel
    np.testing.assert_array_equal(got_slot[valid], o_row_slot[valid])
    return seg


@pytest.mark.parametrize("R,E", [(32768, 64), (32768, 8), (65536, 64), (524288, 128), (1, 128), (2, 2), (1000, 1), (4097, 72), (8, 4096),
                                  (65537, 64), (100000, 8), (40000, 800), (40000, 900)])
@pytest.mark.parametrize("align", [128, 256])
@pytest.mark.parametrize("dtype", [torch.int32, torch.long])
def test_sort_by_expert_matches_oracle(device, R, E, align, dtype):
    g = torch.Generator().manual_seed(R + E)
    ids = torch.randint(0, E, (R,), generator=g, dtype=dtype)
    _check_sort(device, ids, E, align)


def test_sort_empty_experts_zipf_and_golden(device):
    ids = torch.from_numpy(GOLDEN["small_ids"])
    E = int(GOLDEN["small_num_experts"][0])
    seg = _check_sort(device, ids, E, 128)
    np.testing.assert_array_equal(seg.sorted_scattered_idxs.cpu().numpy(), GOLDEN["small_sorted_scattered_idxs"])
    np.testing.assert_array_equal(seg.sorted_expert_idxs.cpu().numpy(), GOLDEN["small_sorted_expert_idxs"])
    # Zipf(1.0)-like load over 8 experts, the C3 routing shape
    p = 1.0 / np.arange(1, 9)
    ids = torch.from_numpy(np.random.default_rng(0).choice(8, size=32768, p=p / p.sum()))
    for _ in range(2):  # second call reuses the self-restoring workspace
        _check_sort(device, ids, 8, 256)
    # all rows to one expert, at the far end
    _check_sort(device, torch.full((5000,), 63, dtype=torch.int32), 64, 128)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,E,k", [(16384, 64, 2), (1000, 128, 8), (1, 8, 2)])
def test_load_balancing_loss_matches_oracle(device, dtype, T, E, k):
    """cute_kernels.load_balancing_loss (continuous_count_cute + softmax_cute) against the one-hot formulation in the
    oracle: value and gradient w.r.t. the router logits. fp32 1e-5; bf16: the probabilities are rounded to bf16 before
    the mean (rtol 1e-2)."""
    from oracle import moe_oracle as mo

    g = torch.Generator().manual_seed(E + k)
    logits = torch.randn(T, E, generator=g).to(dtype)
    sel = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(min(T, 64))])
    sel = sel.repeat((T + sel.size(0) - 1) // sel.size(0), 1)[:T]
    lg = logits.clone().to(device).requires_grad_()
    loss = cute_kernels.load_balancing_loss(lg, sel.to(device))
    loss.backward()
    lo = logits.clone().float().requires_grad_()
    want = mo.load_balancing_loss_torch(lo, sel)
    want.backward()
    tol = dict(rtol=1e-5, atol=1e-6) if dtype == torch.float32 else dict(rtol=1e-2, atol=1e-3)
    torch.testing.assert_close(loss.cpu(), want.detach(), **tol)
    gtol = dict(rtol=1e-4, atol=1e-7) if dtype == torch.float32 else dict(rtol=5e-2, atol=2e-4 / max(T, 1) + 1e-6)
    torch.testing.assert_close(lg.grad.float().cpu(), lo.grad, **gtol)
    f, P = cute_kernels.load_balancing_stats(lg.detach(), sel.to(device))
    assert abs(float(f.sum()) - k) < 1e-5 and abs(float(P.sum()) - 1.0) < 1e-2


def test_sort_by_expert_out_of_range_ids_are_dropped_and_can_be_detected(device):
    """The contract for ids outside [0, E): dropped from counts and offsets (ends[-1] < R), the rest sorted as if they
    were not there; validate=True turns that into an error."""
    ids = torch.tensor([3, 0, 7, 2, 2, -1, 1, 0, 9, 3], dtype=torch.int32)
    E = 4
    seg = cute_kernels.sort_by_expert(ids.to(device), E, 128)
    keep = (ids >= 0) & (ids < E)
    want_counts = torch.bincount(ids[keep].long(), minlength=E)
    assert seg.counts.cpu().long().tolist() == want_counts.tolist()
    placed = int(seg.ends[-1])
    assert placed == int(keep.sum()) < ids.numel()
    order = [i for e in range(E) for i in range(ids.numel()) if int(ids[i]) == e]  # stable sort of the valid ids
    assert seg.sorted_scattered_idxs[:placed].cpu().tolist() == order
    assert seg.sorted_expert_idxs[:placed].cpu().tolist() == sorted(ids[keep].tolist())
    with pytest.raises(ValueError, match="outside"):
        cute_kernels.sort_by_expert(ids.to(device), E, 128, validate=True)
    cute_kernels.sort_by_expert(ids[keep].to(device), E, 128, validate=True)  # all in range: no error


@pytest.mark.parametrize("R,E", [(1, 1), (63, 2), (65, 60), (1023, 8), (1025, 512), (2049, 128), (4096, 64), (4096, 513), (4097, 64)])
@pytest.mark.parametrize("align", [16, 256])
@pytest.mark.parametrize("dtype", [torch.int32, torch.long])
def test_sort_of_few_ids_in_one_block(device, R, E, align, dtype):
    """Both sides of the lines (ids, experts) up to which one block does the whole sort, skewed so that waves meet runs of one
    id and some experts stay empty; and the same ids with some out of range, which both forms drop."""
    g = torch.Generator().manual_seed(R + E)
    ids = (torch.rand(R, generator=g) ** 3 * E).to(dtype).clamp_(max=E - 1)
    _check_sort(device, ids, E, align)
    ids[::3] = torch.tensor([-1, E, 2**31 - 1], dtype=dtype).repeat(R)[: ids[::3].numel()]
    seg = cute_kernels.sort_by_expert(ids.to(device), E, align)
    kept = ((ids >= 0) & (ids < E)).nonzero().flatten()
    order = kept[torch.sort(ids[kept], stable=True).indices]
    assert int(seg.ends[-1]) == order.numel()
    assert torch.equal(seg.sorted_scattered_idxs.cpu()[: order.numel()].long(), order)
    assert torch.equal(seg.counts.cpu().long(), torch.bincount(ids[kept].long(), minlength=E))


# where one block hands over to two launches: 3,072 ids over more than 384 experts, 4,096 over fewer
@pytest.mark.parametrize("R,E", [(4096, 129), (4097, 129), (4096, 384), (4097, 384), (3072, 385), (3073, 385), (3072, 512), (3073, 512), (4096, 128)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.long])
def test_sort_on_both_sides_of_one_block(device, R, E, dtype):
    test_sort_of_few_ids_in_one_block(device, R, E, 64, dtype)


@pytest.mark.parametrize("R,E", [(5121, 60), (4099, 512), (4099, 513), (66000, 1), (262145, 512), (131073, 384), (20001, 4096), (300001, 128)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.long])
def test_sort_over_many_blocks(device, R, E, dtype):
    """Two launches: a ragged last block and one with no ids left, both widths of block (to 512 bins and beyond), bins that do
    not divide the block, the most blocks that the table of counts allows, and segments longer than the registers hold."""
    test_sort_of_few_ids_in_one_block(device, R, E, 128, dtype)


# a bin per lane, two, and the kernels for any number; one block and several; counts of no, one and several rounds of 256 ids a wave
@pytest.mark.parametrize("E", [63, 64, 65, 127, 128, 129])
@pytest.mark.parametrize("R", [1, 4095, 4096, 4097, 70000, 600001])
def test_sort_by_bins_per_lane(device, R, E):
    g = torch.Generator().manual_seed(R + E)
    ids = torch.randint(-1, E + 1, (R,), generator=g, dtype=torch.int32)  # ids outside [0, E) are dropped
    ids[ids == 5] = 6
    seg = cute_kernels.sort_by_expert(ids.to(device), E, 64)
    kept = torch.nonzero((ids >= 0) & (ids < E)).flatten()
    order = kept[torch.sort(ids[kept], stable=True)[1]]
    counts = torch.bincount(ids[kept].long(), minlength=E)
    n = kept.numel()
    assert torch.equal(seg.counts.cpu().long(), counts) and torch.equal(seg.ends.cpu().long(), counts.cumsum(0))
    assert torch.equal(seg.sorted_scattered_idxs.cpu()[:n].long(), order)
    assert torch.equal(seg.sorted_expert_idxs.cpu()[:n], ids[order])
    padded = (counts + 63) // 64 * 64
    starts = torch.cat((torch.zeros(1, dtype=torch.long), padded.cumsum(0)))
    assert torch.equal(seg.seg_starts.cpu().long(), starts)
    rows = torch.arange(n) - (counts.cumsum(0) - counts)[ids[order].long()] + starts[ids[order].long()]
    assert torch.equal(seg.row_slot.cpu().long()[rows], order)
    tiles = torch.repeat_interleave(torch.arange(E), padded // 64)
    owners = seg.tile_expert.cpu().long()
    assert torch.equal(owners[: tiles.numel()], tiles) and bool((owners[tiles.numel() :] == -1).all())
