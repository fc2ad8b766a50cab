"""The work that a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values. `listed()` names the fixed cases, `draw(rng)` gives further ones of the same ranges,
`prepare(case, seed)` makes what a program has in hand before the call, `run(state)` is one pass through the public entry
points, `work(case)` what a pass cannot do without, `tolerance(case)` how far two correct implementations may lie apart.

Kinds of case
  moe       one MoE layer: inference forward (no_grad) or a training step's forward + backward, with or without the RMSNorm
            ahead of it
  moe_e4m3  the quantised-expert layer behind its RMSNorm (inference only)
  norm      RMSNorm, or the residual add fused with it: forward + backward
  swiglu    the stand-alone packed SwiGLU: forward + backward
  routing   top-k routing of router logits and the stable sort of the routed rows by expert
  count     the histogram of expert ids
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "cute-kernels_amd"))  # imported from the root of the tree that is measured
import cute_kernels as ck  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
EPS = 1e-6


def _moe(name, T, E, k, H, I, train, norm=False, dtype="bf16", act="swiglu", bias=False, zipf=0.0):
    case = {"kind": "moe", "tokens": T, "experts": E, "top_k": k, "hidden": H, "inter": I, "train": train, "norm": norm,
            "dtype": dtype, "act": act, "bias": bias, "zipf": zipf}
    return dict(case, name=name) if name else case


def _e4m3(name, T, E, k, H, I, zipf=0.8):
    case = {"kind": "moe_e4m3", "tokens": T, "experts": E, "top_k": k, "hidden": H, "inter": I, "dtype": "bf16", "zipf": zipf}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one decoding step of a server: 8 sequences through the Mixtral-shape layer (8 wide experts). Nearly every expert's
        # weights are read for two rows each
        _moe("decode_mixtral", 8, 8, 2, 4096, 14336, train=False, zipf=1.0),
        # one decoding step of 64 sequences through the fine-grained layer (64 narrow experts, top-8) behind its norm
        _moe("decode_fine", 64, 64, 8, 2048, 1408, train=False, norm=True),
        # one decoding step of 128 sequences through the quantised-expert layer (128 experts, top-8)
        _e4m3("decode_e4m3", 128, 128, 8, 4096, 1536),
        # prompts of a few requests, 2,000 tokens in all: ordinary prefill through the Mixtral-shape layer
        _moe("prefill_mixtral", 2000, 8, 2, 4096, 14336, train=False, zipf=1.0),
        # a training step on a small micro-batch of the layer form with biases and the tanh GELU, in fp16
        _moe("train_gelu_bias", 1500, 16, 4, 1536, 4096, train=True, dtype="fp16", act="gelu", bias=True),
        # a training step of the fine-grained layer behind its norm: many small ragged segments
        _moe("train_fine", 8192, 64, 8, 2048, 1408, train=True, norm=True),
        # a training step of the Mixtral-shape layer: the largest case
        _moe("train_mixtral", 16384, 8, 2, 4096, 14336, train=True, zipf=1.0),
        # offline / prefill batch through the quantised-expert layer
        _e4m3("batch_e4m3", 65536, 128, 8, 4096, 1536),
        # the step ahead of every block of a transformer in training: residual add + RMSNorm, forward and backward
        {"name": "residual_norm", "kind": "norm", "residual": True, "rows": 16384, "hidden": 4096, "dtype": "bf16"},
        # the dense MLP's activation in training, forward and backward
        {"name": "swiglu_packed", "kind": "swiglu", "rows": 4099, "inter": 5632, "dtype": "bf16"},
        # the router's bookkeeping of one batch: top-2 of 64 experts and the stable sort of 32,768 routed rows
        {"name": "routing", "kind": "routing", "tokens": 16384, "experts": 64, "top_k": 2, "dtype": "bf16"},
        # load statistics of a batch's expert ids
        {"name": "count", "kind": "count", "ids": 1 << 22, "experts": 64, "long": False},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm: odd ones as likely as even ones."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


# layer shapes (experts, top-k, hidden, intermediate) of the framework's own configurations
_SHAPES = ((8, 2, 4096, 14336), (64, 8, 2048, 1408), (128, 8, 4096, 1536))
_LARGEST_WEIGHTS = 3 * 128 * 4096 * 1536
_LARGEST_FLOPS = 18.0 * 16384 * 2 * 4096 * 14336


def _layer_shape(rng):
    if rng.random() < 0.6:
        return rng.choice(_SHAPES)
    E = rng.choice((8, 16, 32, 64, 128))
    H, I = 128 * rng.randint(6, 32), 32 * rng.randint(16, 176)
    while 3 * E * H * I > _LARGEST_WEIGHTS:
        I = 32 * max(1, I // 64)
    return E, rng.choice((1, 2, 4, 6, 8)), H, I


def draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "train", "train", "e4m3", "e4m3", "norm", "swiglu", "routing", "count"))
    if kind in ("decode", "prefill", "train"):
        E, k, H, I = _layer_shape(rng)
        train = kind == "train"
        per_token = (18.0 if train else 6.0) * k * H * I
        lo, hi = {"decode": (1, 256), "prefill": (257, 16384), "train": (128, 16384)}[kind]
        T = _log(rng, lo, min(hi, int(_LARGEST_FLOPS / per_token)))
        act = rng.choice(("swiglu", "swiglu", "swiglu", "gelu"))
        return _moe(None, T, E, k, H, I, train=train, norm=rng.random() < 0.5, dtype=rng.choice(("bf16", "bf16", "fp16")),
                    act=act, bias=act == "gelu" and rng.random() < 0.5, zipf=rng.choice((0.0, 0.8, 1.0)))
    if kind == "e4m3":
        E, k, H, I = _layer_shape(rng)
        H, I = 128 * (H // 128), 128 * max(1, I // 128)
        T = _log(rng, 1, min(65536, int(_LARGEST_FLOPS / (6.0 * k * H * I))))
        return _e4m3(None, T, E, k, H, I, zipf=rng.choice((0.0, 0.8)))
    if kind == "norm":
        return {"kind": "norm", "residual": rng.random() < 0.5, "rows": _log(rng, 1, 65536), "hidden": 64 * rng.randint(8, 96),
                "dtype": rng.choice(("bf16", "bf16", "fp16", "fp32"))}
    if kind == "swiglu":
        return {"kind": "swiglu", "rows": _log(rng, 1, 32768), "inter": 8 * rng.randint(64, 1792),
                "dtype": rng.choice(("bf16", "bf16", "fp16", "fp32"))}
    if kind == "routing":
        E = rng.choice((8, 16, 32, 64, 128))
        return {"kind": "routing", "tokens": _log(rng, 1, 65536), "experts": E, "top_k": rng.choice((1, 2, 4, 6, 8)),
                "dtype": rng.choice(("bf16", "fp16", "fp32"))}
    return {"kind": "count", "ids": _log(rng, 1024, 1 << 26), "experts": rng.choice((8, 16, 60, 64, 128)), "long": rng.random() < 0.5}


# ---------------------------------------------------------------------------------------------------------------
def _tokens(case, gate_weight, g, dtype):
    """Token rows as a trained router meets them: noise that leans towards the token's own experts, which are drawn from
    the case's load (Zipf with exponent `zipf`). A logit's lead of 8 to 10 over the noise of all others, N(0, 1), keeps the
    selection clear; on pure noise every hundredth token has its k-th and (k+1)-th logit within one step of the 16-bit
    type, and two correct implementations choose differently."""
    T, E, k, H = case["tokens"], case["experts"], case["top_k"], case["hidden"]
    dev = gate_weight.device
    load = 1.0 / torch.arange(1, E + 1, device=dev, dtype=torch.float32) ** case["zipf"]
    chosen = torch.multinomial(load.expand(T, E), k, generator=g)
    lean = torch.zeros(T, E, device=dev).scatter_(1, chosen, 8.0 + 2.0 * torch.rand(T, k, device=dev, generator=g))
    w = gate_weight.float()
    x = torch.randn(T, H, device=dev, generator=g)
    return torch.addmm(x, lean, w / w.square().sum(1, keepdim=True)).to(dtype)


def _layer(case, seed):
    """The layer as a program builds it, weights ~ N(0, 0.02) (0.02 is the width the framework's own workloads use),
    router weights ~ N(0, 1/H)."""
    torch.manual_seed(seed)
    act = ck.swiglu_packed_cute if case.get("act", "swiglu") == "swiglu" else torch.nn.GELU(approximate="tanh")
    glu = case.get("act", "swiglu") == "swiglu"
    with torch.device("cuda"):
        moe = ck.MoE(case["experts"], case["top_k"], case["hidden"], case["inter"], act, glu, case.get("bias", False), 0.02)
    with torch.no_grad():
        moe.gate.weight.normal_(0.0, case["hidden"] ** -0.5)
        if case.get("bias"):
            moe.c_fc.bias.normal_(0.0, 0.02)
            moe.c_proj.bias.normal_(0.0, 0.02)
    return moe.to(DTYPES[case["dtype"]])


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES.get(case.get("dtype"))
    kind = case["kind"]
    if kind in ("moe", "moe_e4m3"):
        moe = _layer(case, seed)
        x = _tokens(case, moe.gate.weight.detach(), g, dt)
        state = {"case": case, "moe": moe, "x": x, "norm_weight": None}
        if kind == "moe_e4m3" or case["norm"]:
            state["norm_weight"] = (1 + 0.02 * torch.randn(case["hidden"], device="cuda", generator=g)).to(dt)
        if kind == "moe_e4m3":
            state["moe"] = ck.MoE_E4M3(moe)
        elif case["train"]:
            state["dy"] = torch.randn(x.shape, device="cuda", generator=g).to(dt)
            x.requires_grad_()
            if case["norm"]:
                state["norm_weight"].requires_grad_()
        return state
    if kind == "norm":
        shape = (case["rows"], case["hidden"])
        state = {"case": case, "w": (1 + 0.02 * torch.randn(shape[1], device="cuda", generator=g)).to(dt).requires_grad_()}
        for name in ("x", "residual") if case["residual"] else ("x",):
            state[name] = torch.randn(shape, device="cuda", generator=g).to(dt).requires_grad_()
        for name in ("dy", "dadded") if case["residual"] else ("dy",):
            state[name] = torch.randn(shape, device="cuda", generator=g).to(dt)
        return state
    if kind == "swiglu":
        x = torch.randn(case["rows"], 2 * case["inter"], device="cuda", generator=g).to(dt).requires_grad_()
        return {"case": case, "x": x, "dy": torch.randn(case["rows"], case["inter"], device="cuda", generator=g).to(dt)}
    if kind == "routing":
        return {"case": case, "logits": torch.randn(case["tokens"], case["experts"], device="cuda", generator=g).to(dt)}
    ids = torch.randint(0, case["experts"], (case["ids"],), device="cuda", generator=g)
    return {"case": case, "ids": ids if case["long"] else ids.to(torch.int32)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "moe":
        moe, x, w = state["moe"], state["x"], state["norm_weight"]
        if not case["train"]:
            with torch.no_grad():
                return moe(x) if w is None else moe.forward_with_norm(x, w, EPS)
        moe.zero_grad(set_to_none=True)
        x.grad = None
        if w is not None:
            w.grad = None
        y, logits = moe(x) if w is None else moe.forward_with_norm(x, w, EPS)
        y.backward(state["dy"])
        return [y.detach(), logits.detach(), x.grad, None if w is None else w.grad] + [p.grad for p in moe.parameters()]
    if kind == "moe_e4m3":
        return state["moe"].forward_with_norm(state["x"], state["norm_weight"], EPS)
    if kind == "norm":
        x, w = state["x"], state["w"]
        x.grad = w.grad = None
        if not case["residual"]:
            y = ck.rmsnorm_cute(x, w, EPS)
            y.backward(state["dy"])
            return y.detach(), x.grad, w.grad
        residual = state["residual"]
        residual.grad = None
        y, added = ck.fused_residual_add_rmsnorm_cute(x, residual, w, EPS)
        torch.autograd.backward((y, added), (state["dy"], state["dadded"]))
        return y.detach(), added.detach(), x.grad, residual.grad, w.grad
    if kind == "swiglu":
        x = state["x"]
        x.grad = None
        y = ck.swiglu_packed_cute(x)
        y.backward(state["dy"])
        return y.detach(), x.grad
    if kind == "routing":
        with torch.no_grad():
            gates, selected = ck.route_topk_softmax(state["logits"], case["top_k"], long_indices=False)
            seg = ck.sort_by_expert(selected, case["experts"])
        return gates, selected, seg.sorted_expert_idxs, seg.sorted_scattered_idxs, seg.counts, seg.ends, seg.starts
    return ck.continuous_count_cute(state["ids"], case["experts"])


def _experts_read(case):
    """Experts that at least one of the tokens' slots reaches, on average, if a token's k experts were drawn one by one."""
    load = [1.0 / (e + 1) ** case["zipf"] for e in range(case["experts"])]
    total = sum(load)
    slots = case["tokens"] * case["top_k"]
    reached = sum(1.0 - (1.0 - p / total) ** slots for p in load)
    return max(reached, min(case["top_k"], case["experts"]))


def work(case):
    kind = case["kind"]
    s = torch.empty(0, dtype=DTYPES.get(case.get("dtype"), torch.int32)).element_size()
    if kind in ("moe", "moe_e4m3"):
        T, E, k, H, I = (case[n] for n in ("tokens", "experts", "top_k", "hidden", "inter"))
        matrices = 2 if case.get("act", "swiglu") != "swiglu" else 3
        per_expert = matrices * H * I
        read = _experts_read(case) * per_expert
        rows = T * H * s
        flops = 2.0 * T * k * per_expert + 2.0 * T * E * H
        gate = E * H * s + T * E * s
        if kind == "moe_e4m3":
            return {"bytes": 2 * rows + gate + read, "flops": flops}
        if not case["train"]:
            return {"bytes": 2 * rows + gate + read * s, "flops": flops}
        # forward: x, weights -> y; backward: x, dy, weights -> dx and a gradient for every weight
        return {"bytes": 5 * rows + 3 * gate + (2 * read + E * per_expert) * s, "flops": 3 * flops}
    if kind == "norm":
        n = case["rows"] * case["hidden"] * s
        # with the residual: x, residual -> y, sum; sum, dy, dsum -> two gradients. Without: x -> y; x, dy -> dx
        return {"bytes": (9 if case["residual"] else 5) * n, "flops": 0}
    if kind == "swiglu":
        return {"bytes": 8 * case["rows"] * case["inter"] * s, "flops": 0}
    if kind == "routing":
        T, E, k = case["tokens"], case["experts"], case["top_k"]
        return {"bytes": T * E * s + T * k * (s + 4) + 2 * 4 * T * k + 12 * E, "flops": 0}
    return {"bytes": case["ids"] * (8 if case["long"] else 4) + 4 * case["experts"], "flops": 0}


def tolerance(case):
    """Measured against the same path with 32-bit (layers) or 64-bit (norm, swiglu) tensors throughout: bf16 layers are off
    by 0.7 to 1.5 % (the rounding of logits and gates dominates), fp16 layers by 0.14 %, the quantised layer by 2.2 % (a
    last-bit difference ahead of an e4m3 rounding moves a value by 6 %), norm and swiglu in bf16 by 0.25 %."""
    if case["kind"] == "count":
        return "exact"
    if case["kind"] == "moe_e4m3":
        return {"rel": 3e-2}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if case["kind"] == "moe":
        return {"rel": 2e-2 if case["dtype"] == "bf16" else 6e-3}
    return {"rel": 8e-3 if case["dtype"] == "bf16" else 1.5e-3}
