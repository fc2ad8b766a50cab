"""What the native host module refuses before it looks at a device: shapes the kernels would read or write past."""

import copy
import os
import pickle
import subprocess
import sys
import threading

import pytest
import torch

import cute_kernels as ck
from cute_kernels import _C, scattermoe


def _segments(rows, experts, align=128):
    max_rows = _C.lib().ck_sort_max_rows(rows, experts, align)
    i32 = lambda n: torch.zeros(n, dtype=torch.int32)
    return scattermoe.ExpertSegments(
        i32(rows), i32(rows), i32(experts), i32(experts), i32(experts), i32(experts + 1), i32(max_rows), i32(max_rows // align),
        max_rows, experts, align,
    )


E, T, k, H, I = 4, 6, 2, 64, 128
bf16 = dict(dtype=torch.bfloat16)
X, GATES = torch.zeros(T, H, **bf16), torch.zeros(T, k, **bf16)
W_FC, W_PROJ = torch.zeros(E, 2 * I, H, **bf16), torch.zeros(E, H, I, **bf16)
W8 = [torch.zeros(E, 2 * I, H, dtype=torch.float8_e4m3fn), torch.zeros(E, 2 * I), torch.zeros(E, H, I, dtype=torch.float8_e4m3fn), torch.zeros(E, H)]


def test_matching_shapes_get_as_far_as_the_device():
    seg = _segments(T * k, E)
    for call in (
        lambda: scattermoe.swiglu_experts(X, W_FC, W_PROJ, GATES, seg),
        lambda: scattermoe.experts_down(torch.zeros(seg.max_rows, I, **bf16), W_PROJ, GATES, seg),
        lambda: ck.swiglu_experts_e4m3(X, *W8, GATES, _segments(T * k, E, 256)),
        lambda: ck.route_topk_softmax(torch.zeros(T, E), k),
    ):
        with pytest.raises(RuntimeError, match="GPU only"):
            call()


@pytest.mark.parametrize("x", [X.view(2, 3, H), X[0]])
def test_token_rows_are_a_matrix(x):
    with pytest.raises(ValueError):
        scattermoe.swiglu_experts(x, W_FC, W_PROJ, GATES, _segments(T * k, E))
    with pytest.raises(ValueError):
        ck.swiglu_experts_e4m3(x, *W8, GATES, _segments(T * k, E, 256))
    if x.dim() == 3:  # the forward of one linear reads rows only; its backward writes an [T, K] gradient
        with pytest.raises(ValueError):
            _C.host().experts_up_backward(
                torch.zeros(640, 2 * I, **bf16), x, W_FC, None, _segments(T * k, E), k, True, False, False, scattermoe._flags()
            )


def test_gates_and_weights_have_their_dimensions():
    seg = _segments(T * k, E)
    h = torch.zeros(seg.max_rows, I, **bf16)
    for gates in (GATES.flatten(), GATES.view(2, 3, k)):
        with pytest.raises(ValueError):
            scattermoe.swiglu_experts(X, W_FC, W_PROJ, gates, seg)
        with pytest.raises(ValueError):
            scattermoe.experts_down(h, W_PROJ, gates, seg)
        with pytest.raises(ValueError):
            ck.swiglu_experts_e4m3(X, *W8, gates, _segments(T * k, E, 256))
    for w_fc, w_proj in ((W_FC.flatten(0, 1), W_PROJ), (W_FC, W_PROJ.flatten(0, 1))):
        with pytest.raises(ValueError):
            scattermoe.swiglu_experts(X, w_fc, w_proj, GATES, seg)
    with pytest.raises(ValueError):
        scattermoe.experts_down(h, W_PROJ.flatten(0, 1), GATES, seg)
    with pytest.raises(ValueError):
        scattermoe.experts_up(X, W_FC.flatten(0, 1), seg, k)


@pytest.mark.parametrize("shape", [(E,), (2, 3, E)])
def test_router_logits_are_a_matrix(shape):
    with pytest.raises(ValueError):
        ck.route_topk_softmax(torch.zeros(shape), 2)


def test_gates_can_be_copied_and_saved(tmp_path):
    """The router's gates carry a slot of the native module as an attribute. It belongs to one backward pass: a copy of the
    gates gets an empty one of its own."""
    gates = torch.rand(3, 2)
    gates._ck_gate_slot = _C.host().GateSlot()
    gates._ck_gate_slot.d_gates_f32 = torch.ones(3, 2)
    torch.save(gates, tmp_path / "gates.pt")
    for other in (copy.deepcopy(gates), pickle.loads(pickle.dumps(gates)), torch.load(tmp_path / "gates.pt", weights_only=False)):
        assert torch.equal(other, gates)
        slot = other._ck_gate_slot
        assert type(slot) is type(gates._ck_gate_slot) and slot is not gates._ck_gate_slot and slot.d_gates_f32 is None
    assert gates._ck_gate_slot.d_gates_f32 is not None
    # another process finds the class where the package is on its path
    load = "import pickle, sys; print(type(pickle.load(sys.stdin.buffer)._ck_gate_slot).__module__)"
    env = dict(os.environ, PYTHONPATH=os.path.dirname(os.path.dirname(_C.__file__)))
    out = subprocess.run([sys.executable, "-c", load], input=pickle.dumps(gates), capture_output=True, env=env, timeout=100)
    assert out.stdout.split() == [b"cute_kernels._ck_host"], out.stderr.decode()


class _Timer:
    def __init__(self):
        self.names = []

    def time(self, name, dims, launch):
        self.names.append((name, dims))
        launch()


def test_launch_timer_may_be_taken_off_while_another_thread_launches():
    """Every launch happens once, with the timer or without: a thread that saw a timer and then waited for the interpreter lock
    finds out whether it is still there."""
    host, launched = _C.host(), []
    timer = _Timer()
    host.set_launch_timer(timer)
    host.timed_without_lock("gemm", 2, 3, lambda: launched.append(0))
    host.set_launch_timer(None)
    host.timed_without_lock("gemm", 2, 3, lambda: launched.append(0))
    assert timer.names == [("gemm", (2, 3))] and len(launched) == 2
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        for i in range(2000):
            host.set_launch_timer(_Timer())
            thread = threading.Thread(target=host.timed_without_lock, args=("gemm", 2, 3, lambda: launched.append(i)))
            thread.start()
            host.set_launch_timer(None)
            thread.join()
    finally:
        sys.setswitchinterval(interval)
        host.set_launch_timer(None)
    assert len(launched) == 2002


@pytest.mark.parametrize("rows,hidden,experts,pays", [(100_000, 4096, 64, True), (16384, 4096, 128, True), (16385, 4096, 128, False), (65536, 2560, 128, False),
                                                       (1, 4096, 64, True), (513, 4096, 128, False), (2048, 4096, 96, False), (2049, 2560, 128, True)])
def test_where_the_one_pass_norm_and_router_pays(rows, hidden, experts, pays):
    from cute_kernels.rmsnorm_route import rmsnorm_route_pays

    x = torch.empty(rows, hidden, dtype=torch.bfloat16, device="meta")
    assert rmsnorm_route_pays(x, torch.empty(experts, hidden, dtype=torch.bfloat16, device="meta")) == pays
