"""Performance cases of the MoE layer: what a program that uses this package has it do, over the range of real use.

A case names the entry points it calls ("kind") and the sizes: T tokens, H hidden size, E experts, K experts per
token, I intermediate size; "skew" makes the gate prefer the low experts (Zipf), as trained gates do.

    layer     ops.moe_layer: MoeRoutingTopK, MoeExpertFFN, MoeCombine one after the other (the reference's chain)
    fused     ops.moe_layer_fused: the whole layer in one library call
    ffn       ops.MoeExpertFFN alone, on ids and weights a router of the caller's chose, no workspace given
    ffn_comb  ops.MoeExpertFFNCombine, on ids and weights a router of the caller's chose
    routing   ops.MoeRoutingTopK alone
    combine   ops.MoeCombine alone

All tensors are fp16 (ids int32), the only types the operators take.
"""
from __future__ import annotations

import importlib
import math

import torch

_PKG = "implementing-moe-architecture-operators-on-cann-platform_amd"
ops = importlib.import_module(f"{_PKG}.ops")
synth = importlib.import_module(f"{_PKG}.synth")

_FFN_KINDS = ("layer", "fused", "ffn", "ffn_comb")
_MAX_FLOPS = 2.8e12        # a drawn case stays below the largest listed one (2.9 TFLOP)
_MAX_WEIGHT_BYTES = 3.0e9  # and its expert weights near the listed layers' (the DeepSeek-V3-shaped one apart)


def listed():
    return [
        # A unit-test sized layer: every kernel is launch latency, the call's cost is the host path.
        dict(name="layer_tiny", kind="layer", T=8, H=64, E=4, K=2, I=256, skew=False),
        # One user's decode step with many small experts: 6 of 64 experts' weights are read.
        dict(name="decode_T1_E64", kind="fused", T=1, H=2048, E=64, K=6, I=1408, skew=False),
        # The headline decode step (128 concurrent sequences), the three operators as the reference calls them.
        dict(name="decode_T128", kind="layer", T=128, H=2048, E=16, K=2, I=8192, skew=False),
        # A decode batch on few, large experts with a long hidden size.
        dict(name="decode_T40_H4096", kind="fused", T=40, H=4096, E=8, K=2, I=14336, skew=False),
        # A decode batch on 256 experts with a hidden size of 7168: 22.5 GB of weights, most of them active.
        dict(name="decode_T64_E256", kind="fused", T=64, H=7168, E=256, K=8, I=2048, skew=False),
        # A large continuous batch or one chunk of a chunked prefill: between weight streaming and dense GEMMs.
        dict(name="chunk_T1000", kind="ffn_comb", T=1000, H=2048, E=16, K=2, I=8192, skew=False),
        # A short prompt on many small experts, uneven expert loads, odd token count.
        dict(name="prompt_T1531_E64", kind="fused", T=1531, H=2048, E=64, K=6, I=1408, skew=True),
        # The headline prefill, the three operators.
        dict(name="prefill_T8192", kind="layer", T=8192, H=2048, E=16, K=2, I=8192, skew=False),
        # The largest layer: a prefill on few, large experts.
        dict(name="prefill_T4096_H4096", kind="fused", T=4096, H=4096, E=8, K=2, I=14336, skew=False),
        # A long prefill on many small experts with Zipf-skewed loads.
        dict(name="prefill_T16384_E64", kind="fused", T=16384, H=2048, E=64, K=6, I=1408, skew=True),
        # The expert FFN alone at sizes that are no multiple of any tile (H and I odd multiples of 32).
        dict(name="ffn_ragged", kind="ffn", T=3001, H=1056, E=24, K=3, I=736, skew=False),
        # The router alone over 256 experts, as a caller with its own expert kernels uses it.
        dict(name="routing_E256", kind="routing", T=4096, H=7168, E=256, K=8, I=2048, skew=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_mult32(rng, lo, hi):
    return max(lo, min(hi, 32 * int(round(_log_int(rng, lo, hi) / 32))))


def draw(rng):
    kind = rng.choice(("layer", "layer", "fused", "fused", "ffn", "ffn_comb", "routing", "combine"))
    while True:
        T = _log_int(rng, 1, 16384)
        E = _log_int(rng, 4, 256)
        H = _log_mult32(rng, 96, 7168)
        I = _log_mult32(rng, 96, 14336)
        K = rng.randint(1, min(8, E))
        if 6.0 * T * K * H * I <= _MAX_FLOPS and 6.0 * E * I * H <= _MAX_WEIGHT_BYTES and T * K * H <= 1 << 28:
            return dict(kind=kind, T=T, H=H, E=E, K=K, I=I, skew=rng.random() < 0.3)


def _normal(shape, sigma, gen):
    return torch.empty(shape, dtype=torch.float16, device="cuda").normal_(0.0, sigma, generator=gen)


def _inputs(case, seed):
    """The case's tensors, from the seed alone: activations N(0, 1); gate, W_gate and W_up N(0, 1/H); W_down
    N(0, 1/I), so every intermediate is of order one."""
    T, H, E, K, I = (case[k] for k in "THEKI")
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = {}
    if case["kind"] == "combine":
        s["expert_out"] = _normal((T, K, H), 1.0, gen)
    else:
        s["x"] = _normal((T, H), 1.0, gen)
    w_gate = torch.empty((H, E), dtype=torch.float32, device="cuda").normal_(0.0, 1.0 / math.sqrt(H), generator=gen)
    if case["skew"]:
        w_gate *= torch.from_numpy(synth.zipf_column_scale(E)).to("cuda", torch.float32)
    s["w_gate"] = w_gate.to(torch.float16)
    if case["kind"] in ("ffn", "ffn_comb", "combine"):
        # the caller's own router: top-K of a softmax over its logits, renormalised
        src = s["x"].float() @ w_gate if "x" in s else torch.randn((T, E), device="cuda", generator=gen)
        p, ids = torch.softmax(src, dim=1).topk(K, dim=1)
        s["ids"] = ids.to(torch.int32).contiguous()
        s["w"] = (p / p.sum(dim=1, keepdim=True)).to(torch.float16).contiguous()
    if case["kind"] in _FFN_KINDS:
        ew = torch.empty((E, 3 * I, H), dtype=torch.float16, device="cuda")
        for e in range(E):  # [3I, H]: W_gate, W_up rows of length H, then W_down as [H, I]
            flat = ew[e].view(-1)
            flat[: 2 * I * H].normal_(0.0, 1.0 / math.sqrt(H), generator=gen)
            flat[2 * I * H:].normal_(0.0, 1.0 / math.sqrt(I), generator=gen)
        s["ew"] = ew
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["kind"], s["K"] = case["kind"], case["K"]
    T, H, E, K, I = (case[k] for k in "THEKI")
    if case["kind"] in ("layer", "ffn_comb"):  # a program keeps the workspace over its calls
        s["workspace"] = torch.empty(max(1, ops.workspace_bytes(T, H, E, K, I)), dtype=torch.uint8, device="cuda")
    elif case["kind"] == "fused":
        s["workspace"] = torch.empty(max(1, ops.layer_workspace_bytes(T, H, E, K, I)), dtype=torch.uint8, device="cuda")
    return s


def run(s):
    kind = s["kind"]
    if kind == "layer":
        y, ids, w, eo = ops.moe_layer(s["x"], s["w_gate"], s["ew"], s["K"], s["workspace"])
    elif kind == "fused":
        y, ids, w, eo = ops.moe_layer_fused(s["x"], s["w_gate"], s["ew"], s["K"], 0, s["workspace"])
    elif kind == "ffn":
        return {"expert_out": ops.MoeExpertFFN(s["x"], s["ids"], s["w"], s["ew"])}
    elif kind == "ffn_comb":
        eo, y = ops.MoeExpertFFNCombine(s["x"], s["ids"], s["w"], s["ew"], 0, s["workspace"])
        return {"expert_out": eo, "y": y}
    elif kind == "routing":
        ids, w = ops.MoeRoutingTopK(s["x"], s["w_gate"], s["K"])
        return {"ids": ids, "weights": w}
    else:
        return {"y": ops.MoeCombine(s["expert_out"], s["ids"], s["w"], s["K"])}
    return {"expert_out": eo, "ids": ids, "weights": w, "y": y}


def work(case):
    """Bytes: every input read once and every output written once, expert weights only of experts that tokens
    reach (in expectation, for evenly spread tokens). The SwiGLU intermediate is not counted."""
    T, H, E, K, I = (case[k] for k in "THEKI")
    S, kind = T * K, case["kind"]
    nbytes = flops = 0.0
    if kind in ("layer", "fused", "routing"):
        nbytes += 2 * T * H + 2 * H * E + 6 * S
        flops += 2.0 * T * H * E
    if kind in _FFN_KINDS:
        active = E * (1.0 - (1.0 - K / E) ** T)
        nbytes += 6.0 * active * I * H + 2 * S * H
        flops += 6.0 * S * H * I
        if kind in ("ffn", "ffn_comb"):
            nbytes += 2 * T * H + 4 * S
    if kind in ("layer", "fused", "ffn_comb"):
        nbytes += 2 * T * H
        flops += 2.0 * S * H
    if kind == "combine":
        nbytes += 2 * S * H + 2 * S + 2 * T * H
        flops += 2.0 * S * H
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """fp16 results of fp32 sums: a value is off by half an fp16 step (2^-11) where the SwiGLU intermediate is
    rounded and again where the result is (measured against exact(): expert_out 2.9e-4, y 4.2e-4, weights 2.5e-4);
    sums in another order change which way some values round. The router's
    ids are ranked by fp32 sums: two experts whose logits agree to ~1e-6 may swap, and a swapped pair of slots
    swaps two whole rows of expert_out, sqrt(4 / (T K)) of its norm for one pair."""
    kind, S = case["kind"], case["T"] * case["K"]
    if kind in ("ffn", "ffn_comb", "combine"):
        return {"rel": 1.5e-3}
    swaps = math.ceil(1e-5 * S) if S >= 1000 else 0
    if kind == "routing":
        return {"rel": 1.5e-3, "differ": 2.0 * swaps / S}
    return {"rel": max(1.5e-3, math.sqrt(4.0 * swaps / S)), "differ": 2.0 * swaps / S}


def exact(case, seed):
    """The same outputs in float64 from the same fp16 inputs, nothing rounded on the way."""
    s, kind, K = _inputs(case, seed), case["kind"], case["K"]
    E, I, H = case["E"], case["I"], case["H"]
    if kind == "combine":
        return {"y": (s["expert_out"].double() * s["w"].double().unsqueeze(2)).sum(dim=1)}
    x = s["x"].double()
    if kind in ("layer", "fused", "routing"):
        p, ids = torch.softmax(x @ s["w_gate"].double(), dim=1).topk(K, dim=1)
        w = p / p.sum(dim=1, keepdim=True)
        if kind == "routing":
            return {"ids": ids.to(torch.int32), "weights": w}
    else:
        ids, w = s["ids"].long(), s["w"].double()
    eo = torch.zeros((case["T"], K, H), dtype=torch.float64, device="cuda")
    for e in range(E):
        t, k = (ids == e).nonzero(as_tuple=True)
        if t.numel() == 0:
            continue
        flat = s["ew"][e].view(-1)
        wg, wu = flat[: I * H].view(I, H).double(), flat[I * H: 2 * I * H].view(I, H).double()
        wd = flat[2 * I * H:].view(H, I).double()
        for a in range(0, t.numel(), 2048):  # bounds the float64 intermediates
            ta, ka = t[a: a + 2048], k[a: a + 2048]
            xe = x[ta]
            g = xe @ wg.t()
            eo[ta, ka] = (g * torch.sigmoid(g) * (xe @ wu.t())) @ wd.t()
    if kind == "ffn":
        return {"expert_out": eo}
    y = (eo * w.unsqueeze(2)).sum(dim=1)
    if kind == "ffn_comb":
        return {"expert_out": eo, "y": y}
    return {"expert_out": eo, "ids": ids.to(torch.int32), "weights": w, "y": y}
