"""MoE expert path: routing, token->expert sort, scattered grouped GEMMs, gated combine -- forward and backward.

Semantics follow cute_kernels/kernels/scattermoe/torch_implementation.py:63-201 (reference oracle) and the autograd
conventions of cute_kernels/kernels/scattermoe/triton_implementation/ops.py:143-292. The data layout does not: rows
are kept in a padded grouped order where every expert's segment starts at a multiple of the GEMM tile height, and the
backward GEMMs consume transposed copies that the producing kernels write as they go, so that every matrix product is
contraction-contiguous on both operands.
"""

from __future__ import annotations

import ctypes
import functools
import math
from dataclasses import dataclass

import torch
from torch.fx.experimental.symbolic_shapes import statically_known_true

from . import _C
from .utils import is_tracing, plain_size

_ops = None  # cute_kernels.compile_ops, set by the package once it is imported (used only while torch.compile traces)


@dataclass
class Options:
    """Switches between forms that compute the same result, for tests and measurements (bench.py sets them from its
    command line). The defaults are what the library runs; nothing reads the environment."""

    gemm_split: bool = True  # the last, partial round of GEMM tiles splits its contraction over the idle CUs
    bias_fused: bool = True  # expert biases join the GEMM's fp32 accumulators (False: their own kernel after the GEMM)
    gemm_nn: bool = True  # input-gradient GEMMs read the weight as stored (False: through a transposed copy)
    dw_rows: bool = True  # weight-gradient GEMMs read row-major operands (False: transposed copies)


options = Options()


def _flags() -> int:
    """options as the native host module takes them (csrc/host/host_ops.cpp: Flags)"""
    return options.gemm_split | options.bias_fused << 1 | options.gemm_nn << 2 | options.dw_rows << 3


# ---------------------------------------------------------------------------------------------------------------
# routing
# ---------------------------------------------------------------------------------------------------------------
def _gate_slot(gates: torch.Tensor):
    """The side channel the router attached to these gates, if any: through it the expert block's backward hands the router's
    its unrounded gate gradient (GateSlot in csrc/host/host_ops.cpp)."""
    return getattr(gates, "_ck_gate_slot", None)


def route_topk_softmax(logits: torch.Tensor, k: int, long_indices: bool = True) -> tuple[torch.Tensor, torch.Tensor]:
    """Top-k over the logits and softmax over the k selected logits in fp32, cast back to logits.dtype
    (torch_implementation.py:122-135). Equal logits: the lowest expert index wins. The indices come back as int64 like
    torch.topk's; long_indices=False keeps the kernel's int32 (what the sort consumes fastest)."""
    if is_tracing():
        gates, selected = _ops.route_topk_softmax(logits, k)
        return gates.to(logits.dtype), (selected.long() if long_indices else selected)
    host = _C.host()
    slot = host.GateSlot()
    gates, selected = host.route(logits, k, long_indices, slot)
    gates._ck_gate_slot = slot  # found again by the expert block that consumes these gates
    return gates, selected


@torch.no_grad()
def route_topk_softmax_raw(logits: torch.Tensor, k: int) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(selected int32 [T, k], gates fp32 [T, k], top-k values [T, k] in logits.dtype), no autograd."""
    _C.require_gpu(logits)
    logits = logits.contiguous()
    T, E = logits.shape
    selected = torch.empty(T, k, dtype=torch.int32, device=logits.device)
    gates = torch.empty(T, k, dtype=torch.float32, device=logits.device)
    values = torch.empty(T, k, dtype=logits.dtype, device=logits.device)
    lib = _C.lib()
    with torch.cuda.device(logits.device):
        _C.check(
            lib.ck_route_topk_softmax(
                _C.ptr(logits), _C.dtype_code(logits.dtype), T, E, k, _C.ptr(selected), _C.ptr(gates), _C.ptr(values),
                _C.stream(),
            )
        )
    return selected, gates, values


# ---------------------------------------------------------------------------------------------------------------
# sort + segments
# ---------------------------------------------------------------------------------------------------------------
@dataclass
class ExpertSegments:
    """Result of the stable sort by expert, in the reference's vocabulary plus the padded grouped layout."""

    sorted_expert_idxs: torch.Tensor  # int32 [R]
    sorted_scattered_idxs: torch.Tensor  # int32 [R]
    counts: torch.Tensor  # uint32 [E]
    ends: torch.Tensor  # uint32 [E]  inclusive prefix sums (the reference's expert_offsets)
    starts: torch.Tensor  # uint32 [E]  exclusive prefix sums
    seg_starts: torch.Tensor  # int32 [E + 1]
    row_slot: torch.Tensor  # int32 [max_rows]
    tile_expert: torch.Tensor  # int32 [max_rows / align]
    max_rows: int
    num_experts: int
    align: int
    # int32 [max_rows]: the sorted position a padded row stands for, i.e. its row in an UNPADDED grouped tensor [R, *]
    # (the reference's grouped_in / grouped_out layout). Only segments_from_sorted fills it.
    row_pos: torch.Tensor | None = None

    def c_struct(self, rows_in: torch.Tensor | None = None, rows_out: torch.Tensor | None = None) -> _C.ck_segments:
        """rows_in: table a gathered input is read through (default row_slot); rows_out: table the scatter epilogue writes
        through (default: the same as rows_in)."""
        rows_in = self.row_slot if rows_in is None else rows_in
        return _C.ck_segments(
            self.seg_starts.data_ptr(),
            self.counts.data_ptr(),
            self.tile_expert.data_ptr(),
            rows_in.data_ptr(),
            self.max_rows,
            self.num_experts,
            self.align,
            None if rows_out is None else rows_out.data_ptr(),
        )

    @property
    def ld_t(self) -> int:
        """Leading dimension of transposed padded-grouped operands."""
        return self.max_rows


# (rows per expert up to which, tile height) of inference batches: 16-bit layers, and the quantised-expert layer, whose next height is 256
SMALL_TILES, SMALL_TILES_E4M3 = ((6, 16), (22, 32), (30, 64)), ((6, 16), (22, 32), (40, 64))


def _zipf_sum(num_experts: int) -> float:
    """sum of e ** -0.8 over e = 1 .. num_experts by Euler and Maclaurin, 0.5 % off for one expert and less beyond; -4.4375 is zeta(0.8)"""
    return 5.0 * num_experts**0.2 - 4.4375 + 0.5 * num_experts**-0.8 - num_experts**-1.8 / 15


def _zipf_tiles(share: float, num_experts: int) -> int:
    """Row tiles of experts whose loads are Zipf(0.8), every expert with some; share: tiles of the first. Those with more than one
    have half a tile of padding each. Without a loop over the experts: a server asks for another number of rows on every call."""
    several = min(num_experts, int(share**1.25))
    return num_experts - several + (int(share * _zipf_sum(several) + 0.5 * several + 0.5) if several else 0)


def _height_of_large_tiles(num_rows: int, num_experts: int, inference: bool, launches: tuple[tuple[int, int, bool], ...]) -> int:
    """256 or 128 rows for 16-bit layers and single linears below 512 rows per expert, by the shorter sum of launches.
    launches: (columns, contraction, input gradient) of every grouped GEMM that depends on the height. An inference layer is
    judged at an even load and at a Zipf(0.8) one together, since the more uneven the load, the fewer experts fit one tile of 128
    rows; a training step, whose heights lie further apart, at the Zipf(0.8) one alone. In us:
      * a round of 256 x 256 tiles takes 1.6 a 64-deep step with all CUs at work, down to 1.15 with few (the chip's power is
        shared by fewer), and 8.5 for its start and stores; a split last round takes an equal part of the steps and 43 for
        the exchange of the parts, and happens where it takes 40 steps or more off that round;
      * contractions that are no multiple of 64 run on the general kernel, 2.1 and 1.6 a step and no split (single launches with
        256 / 32 tiles: 2,848 deep 121 / 97, 2,816 deep 92 / 59);
      * a step of a 128 x 128 tile takes 0.9 alone on a CU, and 1.6 where the first CUs have two to 1.95 where all do (single
        launches with 256, 272 and 512 tiles: 4,096 deep 70, 117 and 138, 2,048 deep 39, 62 and 77);
      * no launch is shorter than its weights' stream, 6.7 TB/s through 256-row tiles, 4.2 through the general kernel's and 3.8 through
        128-row ones; the input gradient of 128-row tiles, or of the general kernel, transposes the weights first, at 4.2 and in 5 more.
    Over 520 inference layers (8 to 128 experts, 256 to 4,096 wide, 256 to 8,900 inside in steps of 32, gated and not, 31 to 500 rows
    per expert, Zipf(0), (0.8) and (1.0) loads) the chosen height is 0.6 % slower than the better one on average, 256 rows throughout
    15 %. (With the general kernel's step as the other's, and 1.75 for a CU with two tiles, layers of 8 experts at 170 to 390 rows were
    up to 36 % slower.) Both sides at Zipf(0.8), 128 against 256 rows: 32 experts of 3,456 x 896 at 94 rows 211 against 161 us, 8 of
    1,152 x 8,896 at 136 rows 234 against 185, 128 of 2,048 x 1,408 at 60 rows 623 against 556; 8 of 3,584 x 832 at 81 rows 60 against
    83, 8 of 1,408 x 3,552 at 168 rows 106 against 123, 8 of 1,664 x 1,088 without a gate at 392 rows 69 against 83.
    Over 500 training steps of such layers from 12 rows on it is 0.1 % slower on average and 7 % at most, 256 rows throughout 3.5 and
    47 %, over 440 single linears 0.5 % forward and 0.1 % with the backward (always 128: 6 and 10 %). (By the kernels whose parts met
    through device-wide fences, 75 us, and with a gated epilogue that did not split, training steps up to 51 % slower.) Both sides: 8
    of 2,048 x 4,096 without a gate at 160 / 192 / 230 rows 498 / 510 / 617 against 401 / 412 / 461, 16 of 1,024 x 2,016 at 16 / 64 rows
    307 / 359 against 276 / 312, 8 of 1,024 x 3,840 at 40 rows 363 against 275, 8 of 3,200 x 1,120 at 400 rows 543 against 419; at 32
    rows 299 against 306, 8 of 1,024 x 1,024 at 96 / 300 rows 162 / 186 against 180 / 200."""
    even_rows, zipf_rows = num_rows / num_experts + 24, num_rows / _zipf_sum(num_experts)
    cost = {}
    for height in (128, 256):
        loads = [_zipf_tiles(zipf_rows / height, num_experts)]
        if inference:
            loads.append(num_experts * math.ceil(even_rows / height))
        total = 0.0
        for columns, contraction, input_gradient in launches:
            column_tiles, steps, general = -(-columns // height), -(-contraction // 64), contraction % 64 != 0
            megabytes = num_experts * columns * contraction * 2e-6
            if input_gradient and (height == 128 or general):
                total += 2 * megabytes / 4.2 + 5.0
            if height == 128:
                stream = megabytes / 3.8
                for rows in loads:
                    pairs, left = divmod(rows * column_tiles, 512)
                    time = steps * (1.95 * pairs + (0.0 if left == 0 else 0.9 if left <= 256 else 1.25 + left * (0.35 / 256)))
                    total += time if time > stream else stream
                continue
            few, all_cus, stream = (1.6, 2.1, megabytes / 4.2) if general else (1.15, 1.6, megabytes / 6.7)
            for rows in loads:
                rounds, left = divmod(rows * column_tiles, 256)
                time = (steps * all_cus + 8.5) * rounds
                if left:
                    last = steps * (few + (all_cus - few) * left / 256) + 8.5
                    if not general and left <= 128 and steps - (part := -(-steps // min(4, 256 // left))) >= 40:
                        last = min(last, all_cus * part + 43.0 - 8.5 * rounds)
                    time += last
                total += time if time > stream else stream
        cost[height] = total
    return 256 if cost[256] < cost[128] else 128


def _plain_tiles(num_rows: int, num_experts: int) -> int:
    return 256 if num_rows >= 512 * num_experts else 128


def _large_tiles(
    num_rows: int, num_experts: int, dtype: torch.dtype | None, inference: bool, launches: tuple[tuple[int, int, bool], ...], many: bool
) -> int:
    if many or dtype is torch.float32 or num_rows >= 512 * num_experts:  # fp32 GEMMs run on 64-row tiles either way
        return _plain_tiles(num_rows, num_experts)
    return _height_of_large_tiles(num_rows, num_experts, inference, launches)


def _layer_tiles(
    num_rows: int, num_experts: int, dtype: torch.dtype | None, inference: bool, widths: tuple[int, int, bool] | None, many: bool
) -> int:
    if dtype is torch.float32 or (widths is None and not inference):
        return _plain_tiles(num_rows, num_experts)
    if inference and not many:
        for rows, align in SMALL_TILES if widths is not None else SMALL_TILES_E4M3:
            if num_rows <= rows * num_experts:
                return align
    if widths is None:
        return 256
    hidden, inter, gated = widths
    c_fc = 2 * inter if gated else inter
    launches = ((c_fc, hidden, False), (hidden, inter, False))
    if not inference:
        launches += ((inter, hidden, True), (hidden, c_fc, True))
    return _large_tiles(num_rows, num_experts, dtype, inference, launches, many)


_large_tiles_kept, _layer_tiles_kept = functools.lru_cache(4096)(_large_tiles), functools.lru_cache(4096)(_layer_tiles)


def _least(known) -> int:
    """The largest of 0 .. 2^48 for which known(value) holds, if it holds below one value and not from there on."""
    low, high = 0, 1 << 48
    while low < high:
        middle = (low + high + 1) // 2
        if known(middle):
            low = middle
        else:
            high = middle - 1
    return low


def _height(rule, kept, num_rows: int, *rest) -> int:
    """A rule of sizes alone, looked up where it has been asked before. A traced row count that stands for many takes part in
    one comparison only (many), so that a graph is compiled for two ranges of it and no more. If the caller has said between what
    bounds it lies, in none, as any comparison that holds for a part of them has the graph refused: one height for all of them,
    that of their geometric mean."""
    if not is_tracing():
        return kept(num_rows, *rest, False)
    if not statically_known_true(num_rows < 1 << 48):
        return rule(num_rows, *rest, True)
    low = _least(lambda v: statically_known_true(num_rows >= v))
    high = (1 << 48) - _least(lambda v: statically_known_true(num_rows <= (1 << 48) - v))
    return rule(low if low == high else math.isqrt(low * high), *rest, False)


def choose_align(
    num_rows: int, num_experts: int, dtype: torch.dtype | None = None, inference: bool = False,
    widths: tuple[int, int, bool] | None = None,
) -> int:
    """Tile height of the padded layout.
    A caller that says no more than the sizes, and every fp32 layer: 256 rows from 512 rows per expert on, else 128, which
    keeps the padding small.
    widths: (hidden, intermediate, whether the activation is the gated epilogue's) of a 16-bit layer. Below 512 rows per
    expert its GEMMs decide, those of a training step or of the forward alone (_height_of_large_tiles).
    inference (no gradient is asked for): tiles of 16, 32 or 64 rows while the experts average few rows and the load is the
    stream of their weights (grouped_gemm_skinny.hip stages no weights in LDS). An expert of several tiles has its weights
    fetched once per tile, from L2 at best, so the height follows the load. Six gated shapes of 8 to 128 experts, 1,024 to 4,096 wide, at
    3 to 50 rows each and Zipf(0) and (0.8) loads, 156 calls of either layer: the height chosen is 1.1 % (16 bits) and 1.3 % (e4m3) slower
    than the best of 16, 32, 64 and the next one on average (with 14 rows as the end of 32-row tiles and 30 of e4m3's 64-row ones 1.7
    and 3.9). On average over the shapes tiles of 16 / 32 / 64 / 128 rows are at 8 rows 4 / 1 / 11 / 33 % off the best, at 14 16 / 0 / 7 /
    27, at 22 45 / 1 / 4 / 19, at 30 58 / 14 / 1 / 7, at 40 80 / 37 / 3 / 2; the quantised-expert layer's, whose next height is 256, at 8
    rows 4 / 2 / 13 / 53, at 14 15 / 0 / 11 / 44, at 22 39 / 0 / 7 / 29, at 30 44 / 6 / 1 / 16, at 40 58 / 24 / 1 / 7, at 50 76 / 29 / 3 / 3.
    In e4m3, even load, 128 experts of 4,096 x 1,536 at 5 / 8 / 22 / 30 / 40 / 50 rows: tiles of 16 390 / 401 / 774 / 926 / 1,093 / 1,337 us,
    of 32 379 / 394 / 466 / 627 / 891 / 952, of 64 422 / 436 / 515 / 553 / 596 / 646, of 256 571 / 573 / 591 / 600 / 605 / 616; 64 of 2,048 x
    1,408 at 8 / 22 rows: of 16 115 / 197, of 32 111 / 135, of 64 135 / 146."""
    return _height(_layer_tiles, _layer_tiles_kept, num_rows, num_experts, dtype, inference, widths)


def sort_by_expert(
    expert_ids: torch.Tensor, num_experts: int, align: int | None = None, validate: bool = False
) -> ExpertSegments:
    """Stable sort of the flat (token, slot) expert ids, with counts / offsets and the tile-aligned segment tables.

    Contract: every id lies in [0, num_experts) -- what a top-k over num_experts logits produces. An id outside that
    range is dropped, not sorted (the reference's argsort / bincount path would keep it or raise): the counts exclude it,
    ends[-1] falls short of the number of ids, and the last entries of sorted_expert_idxs / sorted_scattered_idxs and
    the row_slot entries nobody owns stay unwritten. validate=True checks ends[-1] against the number of ids and raises
    on a mismatch; it costs a device-to-host read, so the layer does not ask for it."""
    assert expert_ids.dtype in (torch.int32, torch.long)
    if align is None:
        align = _plain_tiles(plain_size(expert_ids.numel()), num_experts)
    if is_tracing():
        return _ops.sort_by_expert_segments(expert_ids, num_experts, align)
    seg = _sort_by_expert_eager(expert_ids, num_experts, align)
    if validate and expert_ids.numel() > 0:
        placed = int(seg.ends[-1])
        if placed != expert_ids.numel():
            raise ValueError(
                f"sort_by_expert: {expert_ids.numel() - placed} of {expert_ids.numel()} expert ids lie outside [0, {num_experts})"
            )
    return seg


def _sort_by_expert_eager(expert_ids: torch.Tensor, num_experts: int, align: int, apart: bool = False) -> ExpertSegments:
    *tables, max_rows = _C.host().sort_by_expert(expert_ids, num_experts, align, apart)
    return ExpertSegments(*tables, max_rows, num_experts, align)


# ---------------------------------------------------------------------------------------------------------------
# thin launch helpers (allocate outputs, pass pointers)
# ---------------------------------------------------------------------------------------------------------------
class LaunchTimer:
    """Optional per-launch timing of the grouped GEMMs with events on the launch stream (used by bench.py).
    records: list of (kernel name, [N, K] or [M, N] of the launch, start event, end event). Names follow the entry point
    and epilogue, so that at the benchmark's shapes one name is one kernel instantiation: grouped_gemm<epilogue>
    (ck_grouped_gemm), grouped_gemm_nn<epilogue> (ck_grouped_gemm_nn, weights read as stored), grouped_gemm<dw>
    (ck_grouped_gemm_dw, transposed operands), grouped_gemm_dw_rows (ck_grouped_gemm_dw_rows, row-major operands)."""

    def __init__(self) -> None:
        self.records: list = []

    def time(self, name: str, dims: tuple, fn) -> None:
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        fn()
        end.record()
        self.records.append((name, dims, start, end))



def set_launch_timer(timer: LaunchTimer | None) -> None:
    """Every expert GEMM launched from now on goes through timer.time (None: no timing)."""
    _C.host().set_launch_timer(timer)


def _split_workspace(device: torch.device) -> torch.Tensor:
    """Workspace of ck_grouped_gemm_ws / ck_grouped_gemm_nn_ws (split last round of tiles) on this device and stream."""
    return _C.host().split_workspace(torch.empty(0, device=device))


def _gemm_f32(a, gather_div, w, w_is_kn: bool, N: int, K: int, seg: ExpertSegments, scatter: bool, y, bias=None,
              rows_in=None, rows_out=None):
    """The grouped GEMMs of fp32 tensors (fp32 MFMA; see ck_grouped_gemm_f32)."""
    _C.host().gemm_f32(a, gather_div, w, w_is_kn, N, K, seg, scatter, y, bias, rows_in, rows_out)


def _gemm(a, gather_div, w, seg: ExpertSegments, epilogue, y, y_t=None, aux=None, aux_in=None, rows_in=None, rows_out=None):
    _C.host().gemm(a, gather_div, w, seg, epilogue, y, y_t, aux, aux_in, rows_in, rows_out, _flags())


def _bias_in_epilogue(seg: ExpertSegments, K: int) -> bool:
    """Whether ck_grouped_gemm takes the per-expert bias as an operand of its grouped / scatter epilogue (the bias joins
    the fp32 accumulators and the output is rounded once, like F.linear). options.bias_fused = False adds it with its
    own kernel after the GEMM instead (two roundings; kept for comparison)."""
    return options.bias_fused


def _fp32(t: torch.Tensor) -> bool:
    """fp32 expert tensors: always the row-major weight-gradient form and the bias in the GEMM's epilogue (the fp32
    kernels have no other form)."""
    return t.dtype == torch.float32


def _gemm_dx(d_y, w, seg: ExpertSegments, epilogue, out, rows_out=None):
    """out = d_y @ w[e] per expert, w [E, out_features, in_features] as the forward stores it: the input-gradient GEMM.
    rows_out: the table a scatter epilogue writes through (default seg.row_slot)."""
    _C.host().gemm_dx(d_y, w, seg, epilogue, out, rows_out, _flags())


def _gemm_dw(a_t, b_t, seg: ExpertSegments, dw):
    _C.host().gemm_dw(a_t, b_t, seg, dw)


def _gemm_dw_rows(a, b, seg: ExpertSegments, dw):
    """dw[e] = a[rows of e]^T @ b[rows of e] from row-major padded-grouped operands (no transposed copies)."""
    _C.host().gemm_dw_rows(a, b, seg, dw)


def _dw_from_rows(align: int, *shapes: tuple[int, int]) -> bool:
    """Whether the weight-gradient GEMMs of shapes (M, N), ... read row-major operands instead of transposed copies
    (csrc/host/host_ops.cpp)."""
    return _C.host().dw_from_rows(align, _flags(), [(int(m), int(n)) for m, n in shapes])


def _group_rows(src, coeff, fan_out, seg: ExpertSegments, want_grouped: bool, want_transposed: bool, rows=None):
    """Padded grouped copy of `src` rows (fan_out == 0: src is already padded-grouped) and / or its transpose. rows: the
    table the rows are read through (default seg.row_slot)."""
    return _C.host().group_rows(src, coeff, fan_out, seg, want_grouped, want_transposed, rows)


def _transpose_weights(w: torch.Tensor) -> torch.Tensor:
    return _C.host().transpose_weights(w)


def _combine(expanded, gates, T, k, H, grad_out=None, want_out=True, want_d_gates=False):
    out = torch.empty(T, H, dtype=expanded.dtype, device=expanded.device) if want_out else None
    d_gates = torch.empty(T, k, dtype=expanded.dtype, device=expanded.device) if want_d_gates else None
    with torch.cuda.device(expanded.device):
        _C.check(
            _C.lib().ck_combine_rows(
                _C.ptr(expanded), _C.ptr(gates), T, k, H, _C.ptr(out), _C.ptr(grad_out), _C.ptr(d_gates),
                _C.dtype_code(expanded.dtype), _C.stream(),
            )
        )
    return out, d_gates


def _gate_grad(expanded, grad_out, T, k, H, gates_dtype, slot):
    """d_gates in fp32 (kept in `slot` for the router's backward) and rounded to the gates' dtype for autograd."""
    assert gates_dtype == expanded.dtype, "gates and expert outputs should have the same dtype"
    return _C.host().gate_grad(expanded, grad_out, T, k, H, slot)


def gather_rows(src: torch.Tensor, idx: torch.Tensor, coeff: torch.Tensor | None = None, fan_out: int = 1) -> torch.Tensor:
    """out[n] = src[idx[n] // fan_out] * coeff[idx[n]] -- the reference's `group` (ops.py:108-140)."""
    _C.require_gpu(src, idx)
    src = src.contiguous()
    out = torch.empty(idx.numel(), src.size(-1), dtype=src.dtype, device=src.device)
    with torch.cuda.device(src.device):
        _C.check(
            _C.lib().ck_gather_rows(
                _C.ptr(src), _C.ptr(idx), _C.ptr(coeff), fan_out, idx.numel(), src.size(-1), _C.ptr(out),
                _C.dtype_code(src.dtype), _C.stream(),
            )
        )
    return out


def _add_expert_bias(y: torch.Tensor, bias: torch.Tensor, seg: ExpertSegments, row_expert: torch.Tensor | None) -> None:
    """y[r] += bias[expert of row r] in place: padded grouped rows (row_expert None) or token-order rows."""
    _C.host().add_expert_bias(y, bias, seg, row_expert)


def _expert_bias_grad(d_y: torch.Tensor, seg: ExpertSegments) -> torch.Tensor:
    """[E, N] column sums of the padded grouped rows of every expert."""
    return _C.host().expert_bias_grad(d_y, seg)


def _slot_experts(seg: ExpertSegments) -> torch.Tensor:
    """Expert of every flat (token, slot) index, int32 [R] (the inverse of the sort)."""
    slot_expert = torch.empty_like(seg.sorted_expert_idxs)
    slot_expert[seg.sorted_scattered_idxs.long()] = seg.sorted_expert_idxs
    return slot_expert


def _check_expert_dtypes(x: torch.Tensor, *weights: torch.Tensor) -> None:
    if x.dtype not in (torch.bfloat16, torch.float16, torch.float32):
        raise NotImplementedError(f"the MI355X expert GEMMs take bf16 / fp16 / fp32 inputs; got {x.dtype}")
    for w in weights:
        assert w.dtype == x.dtype, "expert weights and activations should have the same dtype"
    assert x.size(-1) % 8 == 0, "hidden size should be a multiple of 8"


# ---------------------------------------------------------------------------------------------------------------
# generic expert linears (any activation between them)
# ---------------------------------------------------------------------------------------------------------------
def experts_up(
    x: torch.Tensor, weight: torch.Tensor, seg: ExpertSegments, k: int, bias: torch.Tensor | None = None,
    gelu_tanh: bool = False, down: tuple[torch.Tensor, torch.Tensor, torch.Tensor | None] | None = None,
) -> torch.Tensor:
    """x [T, H] -> c_fc output in padded grouped order [max_rows, N] (+ bias[e] on expert e's rows; pad rows are zero); with
    gelu_tanh, the tanh-approximated GELU of that output, applied in the GEMM's epilogue.
    down: (weight, gates, bias) of the experts_down that follows a gelu_tanh c_fc of a 16-bit layer. Both then are one
    autograd node and the result is experts_down's: nothing outside sees the grouped rows in between, so that neither they
    nor their gradient need zeros in the pad rows."""
    _check_expert_dtypes(x, weight)
    assert bias is None or (bias.dtype == x.dtype and bias.shape == weight.shape[:2]), "bias should be [E, out] in x.dtype"
    if down is not None:
        w_down, gates, bias_down = down
        if is_tracing() or not options.bias_fused:
            return experts_down(experts_up(x, weight, seg, k, bias, gelu_tanh), w_down, gates, seg, bias_down)
        assert gelu_tanh and x.dtype != torch.float32, "only the tanh GELU of a 16-bit layer is one node with its c_proj"
        _check_expert_dtypes(x, w_down)
        assert bias_down is None or (bias_down.dtype == x.dtype and bias_down.shape == w_down.shape[:2]), (
            "bias should be [E, out] in x.dtype"
        )
        return _C.host().gelu_experts(x, weight, w_down, gates.to(x.dtype), bias, bias_down, seg, _gate_slot(gates), _flags())
    if is_tracing():
        op = _ops.experts_up_gelu if gelu_tanh else _ops.experts_up
        out = op(
            x, weight, bias, seg.seg_starts, seg.counts, seg.tile_expert, seg.row_slot, seg.max_rows, seg.num_experts,
            seg.align, k,
        )
        return out[0] if gelu_tanh else out
    return _C.host().experts_up(x, weight, bias, seg, k, gelu_tanh, _flags())


def experts_down(
    h: torch.Tensor, weight: torch.Tensor, gates: torch.Tensor, seg: ExpertSegments, bias: torch.Tensor | None = None
) -> torch.Tensor:
    """h [max_rows, I] (padded grouped) -> sum_k gates * (c_proj output + bias[e]) in token order [T, N]. Pad rows of the
    gradient of h are zero."""
    _check_expert_dtypes(h, weight)
    assert bias is None or (bias.dtype == h.dtype and bias.shape == weight.shape[:2]), "bias should be [E, out] in h.dtype"
    if is_tracing():
        slot_expert = _slot_experts(seg) if bias is not None else None
        return _ops.experts_down(
            h, weight, gates.to(h.dtype), bias, slot_expert, seg.seg_starts, seg.counts, seg.tile_expert, seg.row_slot,
            seg.max_rows, seg.num_experts, seg.align,
        )[0]
    return _C.host().experts_down(h, weight, gates.to(h.dtype), bias, seg, _gate_slot(gates), _flags())


# ---------------------------------------------------------------------------------------------------------------
# fused SwiGLU expert block
# ---------------------------------------------------------------------------------------------------------------
def swiglu_experts(
    x: torch.Tensor, w_fc: torch.Tensor, w_proj: torch.Tensor, gates: torch.Tensor, seg: ExpertSegments,
    act_kind: int = _C.CK_ACT_SWIGLU,
) -> torch.Tensor:
    """Fused expert block for `is_glu=True` (c_fc columns [up | gate]) with `activation_function = swiglu_packed_cute`
    (act_kind CK_ACT_SWIGLU: up * silu(gate)) or `torch.nn.GLU()` (CK_ACT_GLU: up * sigmoid(gate))."""
    _check_expert_dtypes(x, w_fc, w_proj)
    assert x.dtype != torch.float32, "the fused expert block is 16-bit; fp32 layers run experts_up -> activation -> experts_down"
    assert w_fc.size(1) % 16 == 0, "intermediate size should be a multiple of 8"
    if is_tracing():
        grad = torch.is_grad_enabled()
        return _ops.swiglu_experts(
            x, w_fc, w_proj, gates.to(x.dtype), seg.seg_starts, seg.counts, seg.tile_expert, seg.row_slot, seg.max_rows,
            seg.num_experts, seg.align, grad and x.requires_grad, grad and w_fc.requires_grad,
            grad and w_proj.requires_grad, grad and gates.requires_grad, act_kind,
        )[0]
    return _C.host().swiglu_experts(x, w_fc, w_proj, gates.to(x.dtype), seg, act_kind, _gate_slot(gates), _flags())


# ---------------------------------------------------------------------------------------------------------------
# the reference's own expert-linear interface: three index tensors, unpadded grouped rows
# ---------------------------------------------------------------------------------------------------------------
def bincount(x: torch.Tensor, minlength: int) -> torch.Tensor:
    """Histogram of expert ids as the reference's helper returns it (triton_implementation/ops.py:19-28): int64 counts,
    computed by the count kernel (ids outside [0, minlength) are not counted, where torch.bincount would grow or raise)."""
    from .continuous_count import continuous_count_cute

    return continuous_count_cute(x.reshape(-1), minlength).to(torch.int64)


_segments_cache: list = []  # [(sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, versions, align, ExpertSegments)]


@torch.no_grad()
def segments_from_sorted(
    sorted_expert_idxs: torch.Tensor, sorted_scattered_idxs: torch.Tensor, expert_offsets: torch.Tensor,
    align: int | None = None,
) -> ExpertSegments:
    """The padded grouped layout for a sort the caller did: (sorted_expert_idxs, sorted_scattered_idxs) =
    selected_experts.flatten().sort() and expert_offsets = bincount(...).cumsum(-1), the arguments of the reference's
    expert linears (triton_implementation/__init__.py:82-83). One small launch; the result for the last two distinct
    argument triples is kept, so that c_fc and c_proj of one layer call share it."""
    _C.require_gpu(sorted_expert_idxs, sorted_scattered_idxs, expert_offsets)
    assert sorted_expert_idxs.dim() == 1 and sorted_expert_idxs.shape == sorted_scattered_idxs.shape
    assert sorted_expert_idxs.dtype == sorted_scattered_idxs.dtype and sorted_expert_idxs.dtype in (torch.int32, torch.long)
    assert expert_offsets.dim() == 1 and expert_offsets.dtype in (torch.int32, torch.uint32, torch.long)
    R, E = sorted_expert_idxs.numel(), expert_offsets.numel()
    if align is None:
        align = _plain_tiles(R, E)
    tensors = (sorted_expert_idxs, sorted_scattered_idxs, expert_offsets)
    versions = tuple(t._version for t in tensors)
    for entry in _segments_cache:
        if all(a is b for a, b in zip(entry[0], tensors)) and entry[1] == versions and entry[2] == align:
            return entry[3]
    se, ss, off = (t.contiguous() for t in tensors)
    lib = _C.lib()
    dev = se.device
    max_rows = lib.ck_sort_max_rows(R, E, align)
    i32 = dict(dtype=torch.int32, device=dev)
    seg = ExpertSegments(
        sorted_expert_idxs=se, sorted_scattered_idxs=ss, counts=torch.empty(E, dtype=torch.uint32, device=dev), ends=off,
        starts=None, seg_starts=torch.empty(E + 1, **i32), row_slot=torch.empty(max(max_rows, 1), **i32),
        tile_expert=torch.empty(max(max_rows // align, 1), **i32), max_rows=max_rows, num_experts=E, align=align,
        row_pos=torch.empty(max(max_rows, 1), **i32),
    )
    with torch.cuda.device(dev):
        _C.check(
            lib.ck_segments_from_sorted(
                _C.ptr(se), _C.ptr(ss), int(se.dtype == torch.long), _C.ptr(off), int(off.dtype == torch.long), R, E, align,
                _C.ptr(seg.counts), _C.ptr(seg.seg_starts), _C.ptr(seg.row_slot), _C.ptr(seg.row_pos), _C.ptr(seg.tile_expert),
                _C.stream(),
            )
        )
    _segments_cache.insert(0, (tensors, versions, align, seg))
    del _segments_cache[2:]
    return seg


class _ScatteredExperts(torch.autograd.Function):
    """One expert linear on the reference's index tensors (triton_implementation/ops.py:143-292), w [E, N, K] as the
    module stores it. Input rows: token order [T, K] read through sorted_scattered_idxs // k, or (grouped_in) unpadded
    grouped rows [R, K] in sorted order. Output: [R, N] in (token, slot) order, or (grouped_out) in sorted order, or
    (gates [T, fan]) the gated sum over a token's slots [T, N]. The GEMM runs on the padded layout and reads / writes the
    caller's rows through the row tables, so no padded copy of the input or output is made in the forward pass."""

    @staticmethod
    def forward(ctx, x, w, k, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, gates, grouped_in, grouped_out,
                bias=None, gate_slot=None, align=None):
        assert not (gates is not None and grouped_out), "gated outputs are combined per token, not grouped"
        seg = segments_from_sorted(sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, align)
        x = x.contiguous()
        w = w.contiguous()
        E, N, K = w.shape
        R = sorted_expert_idxs.numel()
        assert x.size(-1) == K and x.size(0) == (R if grouped_in else R // k), "input rows do not match the index tensors"
        out = torch.empty(R, N, dtype=x.dtype, device=x.device)
        ctx.seg, ctx.k, ctx.grouped_in, ctx.grouped_out, ctx.gate_slot = seg, k, grouped_in, grouped_out, gate_slot
        if R == 0:  # no routed rows: nothing to launch
            ctx.save_for_backward(x, w, gates, None)
            return out if gates is None else torch.zeros(gates.size(0), N, dtype=x.dtype, device=x.device)
        fused_bias = bias is not None and (_fp32(x) or _bias_in_epilogue(seg, K))
        _gemm(
            x, 1 if grouped_in else k, w, seg, _C.CK_EPI_SCATTER, out, aux_in=bias.contiguous() if fused_bias else None,
            rows_in=seg.row_pos if grouped_in else seg.row_slot, rows_out=seg.row_pos if grouped_out else seg.row_slot,
        )
        if bias is not None and not fused_bias:
            row_expert = sorted_expert_idxs.to(torch.int32) if grouped_out else _slot_experts(seg)
            _add_expert_bias(out, bias.contiguous(), seg, row_expert)
        expanded = None
        if gates is not None:
            gates = gates.contiguous()
            T, fan = gates.shape
            assert T * fan == R, "gates do not match the index tensors"
            expanded = out
            out, _ = _combine(expanded, gates, T, fan, N)
        ctx.save_for_backward(x, w, gates, expanded)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        x, w, gates, expanded = ctx.saved_tensors
        seg, k, grouped_in, grouped_out = ctx.seg, ctx.k, ctx.grouped_in, ctx.grouped_out
        E, N, K = w.shape
        grad_out = grad_out.contiguous()
        need = ctx.needs_input_grad
        need_x, need_w, need_gates = need[0], need[1], need[6]
        need_bias = len(need) > 9 and need[9]
        d_x = d_w = d_gates = d_bias = None
        if seg.sorted_expert_idxs.numel() == 0:  # no routed rows: every gradient is zero
            return (
                torch.zeros_like(x) if need_x else None, torch.zeros_like(w) if need_w else None, None, None, None, None,
                torch.zeros_like(gates) if need_gates and gates is not None else None, None, None,
                torch.zeros(E, N, dtype=w.dtype, device=w.device) if need_bias else None, None, None,
            )
        # the output gradient as padded grouped rows: what both the weight- and the input-gradient GEMM read
        if gates is not None:
            T, fan = gates.shape
            if need_gates:
                d_gates = _gate_grad(expanded, grad_out, T, fan, N, gates.dtype, ctx.gate_slot)
            d_y, _ = _group_rows(grad_out, gates, fan, seg, True, False)
        elif grouped_out:
            d_y, _ = _group_rows(grad_out, None, 1, seg, True, False, rows=seg.row_pos)
        else:
            d_y, _ = _group_rows(grad_out, None, 1, seg, True, False)
        if need_bias:
            d_bias = _expert_bias_grad(d_y, seg)
        if need_w:
            x_g, _ = _group_rows(x, None, 1 if grouped_in else k, seg, True, False, rows=seg.row_pos if grouped_in else None)
            d_w = torch.empty_like(w)
            if _fp32(x) or _dw_from_rows(seg.align, (N, K)):
                _gemm_dw_rows(d_y, x_g, seg, d_w)
            else:
                _, d_y_t = _group_rows(d_y, None, 0, seg, False, True)
                _, x_t = _group_rows(x_g, None, 0, seg, False, True)
                _gemm_dw(d_y_t, x_t, seg, d_w)
        if need_x:
            R = seg.sorted_expert_idxs.numel()
            d_rows = torch.empty(R, K, dtype=x.dtype, device=x.device)
            _gemm_dx(d_y, w, seg, _C.CK_EPI_SCATTER, d_rows, rows_out=seg.row_pos if grouped_in else seg.row_slot)
            d_x = d_rows if grouped_in or k == 1 else _combine(d_rows, None, x.size(0), k, K)[0]
        return d_x, d_w, None, None, None, None, d_gates, None, None, d_bias, None, None


def scattered_experts(
    inputs: torch.Tensor, expert_weights: torch.Tensor, k: int, sorted_expert_idxs: torch.Tensor,
    sorted_scattered_idxs: torch.Tensor, expert_offsets: torch.Tensor, gates: torch.Tensor | None = None,
    grouped_in: bool = False, grouped_out: bool = False, bias: torch.Tensor | None = None,
) -> torch.Tensor:
    """The reference's scattered_experts (triton_implementation/ops.py:295-316), same arguments in the same order:
    expert_weights is the [E, in, out] VIEW `weight.permute(0, 2, 1)` of an [E, out, in] parameter (any other layout is
    copied). `bias` [E, out] is this build's addition (the reference's launcher has none and its module drops the bias)."""
    w = expert_weights.permute(0, 2, 1)  # back to the parameter's own layout: no copy when the argument was the view
    _check_expert_dtypes(inputs, w)
    assert bias is None or (bias.dtype == inputs.dtype and bias.shape == w.shape[:2]), "bias should be [E, out] in x.dtype"
    if gates is not None:
        gates_in = gates
        gates = gates.to(inputs.dtype)
    E, N, K = (plain_size(n) for n in w.shape)
    launches, forward_alone = ((N, K, False),), not (torch.is_grad_enabled() and inputs.requires_grad)
    if not forward_alone:
        launches += ((K, N, True),)
    align = _height(_large_tiles, _large_tiles_kept, plain_size(sorted_expert_idxs.numel()), E, inputs.dtype, forward_alone, launches)
    if is_tracing():
        out = _ops.scattered_experts(
            inputs, w, gates, bias, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, k, grouped_in, grouped_out, align
        )
        return out[0]
    _C.require_gpu(inputs, w, gates, bias, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets)
    return _ScatteredExperts.apply(
        inputs, w, k, sorted_expert_idxs, sorted_scattered_idxs, expert_offsets, gates, grouped_in, grouped_out, bias,
        _gate_slot(gates_in) if gates is not None else None, align,
    )
