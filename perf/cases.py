"""Performance cases of the fused-MoE layer: one pass is one call of the layer on a batch of tokens, hidden states
(and router logits, or the layer's own fp32 gate) in, the combined 16-bit output out.

The shapes are the ones this repository is configured for: a small layer, the Qwen3-30B-A3B layer and the DeepSeek-V3
layer, from one decoding sequence to a full prefill batch, with int8 and int4 weights, uniform and skewed expert
popularity, with and without the shared expert (in line or on its side stream), bf16 and fp16 hidden states, and
weights held as one tensor or as per-expert tensors that a load balancer exchanges."""
from __future__ import annotations

import math

import numpy as np
import torch

from vllm_ascend_amd.fused_moe.contracts import FusedMoEConfig
from vllm_ascend_amd.fused_moe.gate_linear import AscendGateLinear
from vllm_ascend_amd.fused_moe.layer import AscendRoutedExperts
from vllm_ascend_amd.fused_moe.router import AscendFusedTopKRouter
from vllm_ascend_amd.fused_moe.shared_experts import AscendSharedExperts
from vllm_ascend_amd.quantization import get_scheme_class

# hidden size, experts, experts per token, expert width; how the router scores and groups the experts
MODELS = {
    "small": dict(H=1024, E=8, k=2, I=1408, scoring="softmax", groups=1, top_groups=1, factor=1.0),
    "qwen3": dict(H=2048, E=128, k=8, I=768, scoring="softmax", groups=1, top_groups=1, factor=1.0),
    "dsv3": dict(H=7168, E=256, k=8, I=2048, scoring="sigmoid", groups=8, top_groups=4, factor=2.5),
}
W4_GROUP = 256  # weights along K that share an int4 scale


def _case(name, model, tokens, *, weights="int8", dtype="bf16", zipf=0.0, gate=False, shared="no", eplb=False):
    """weights: int8 per channel or int4 in groups; zipf: exponent of the expert popularity (0: uniform); gate: the
    layer computes its logits itself; shared: the shared expert in line ("line") or on its side stream ("side");
    eplb: per-expert weight tensors, and the load of every expert collected for the balancer."""
    c = dict(model=model, tokens=tokens, weights=weights, dtype=dtype, zipf=zipf, gate=gate, shared=shared, eplb=eplb)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one user's chat turn: every launch and every host microsecond is latency between two tokens
        _case("qwen3_decode_1", "qwen3", 1),
        # a serving engine's decode batch: the touched experts' weights stream from HBM
        _case("qwen3_decode_64", "qwen3", 64),
        # a step that mixes decoding sequences with a piece of a prompt, in fp16, router gate inside the layer
        _case("qwen3_mixed_777", "qwen3", 777, dtype="fp16", gate=True),
        # a full prefill batch
        _case("qwen3_prefill_8192", "qwen3", 8192),
        # a small model's batch, few experts and an odd expert width
        _case("small_64", "small", 64),
        # a few sequences on the large layer, shared expert next to the routed ones
        _case("dsv3_decode_3", "dsv3", 3, shared="side"),
        # the large layer's decode batch
        _case("dsv3_decode_64", "dsv3", 64, shared="line"),
        # the large layer's prefill batch with everything the layer owns: gate, routed experts, shared expert
        _case("dsv3_prefill_4096", "dsv3", 4096, gate=True, shared="line"),
        # prompts of one domain: few experts take most of the tokens
        _case("dsv3_zipf_512", "dsv3", 512, zipf=1.1),
        # int4 weights: a decode batch, and a skewed piece of a prompt
        _case("w4a8_decode_16", "dsv3", 16, weights="int4", shared="side"),
        _case("w4a8_zipf_512", "dsv3", 512, weights="int4", zipf=1.1),
        # a layer under a dynamic load balancer: weights exchanged expert by expert, loads collected
        _case("qwen3_eplb_100", "qwen3", 100, zipf=1.1, eplb=True),
    ]


def draw(rng):
    model = rng.choice(["small", "qwen3", "qwen3", "dsv3", "dsv3"])
    weights = "int4" if model == "dsv3" and rng.random() < 0.35 else "int8"
    eplb = weights == "int8" and rng.random() < 0.15
    most = 1024 if weights == "int4" else 2048 if eplb else 4096 if model == "dsv3" else 8192
    tokens = min(most, int(round(math.exp(rng.uniform(0.0, math.log(most + 0.49))))))
    return _case(None, model, tokens, weights=weights, dtype=rng.choice(["bf16", "bf16", "fp16"]),
                 zipf=rng.choice([0.0, 0.0, 1.1]), gate=rng.random() < 0.3,
                 shared=rng.choice(["no", "line", "side"]) if model == "dsv3" else "no", eplb=eplb)


def _fill(out, gen, std, limit):
    """Whole numbers with the bell shape that quantised weights have, a slice at a time (little scratch memory)."""
    for part in out.view(-1).split(1 << 27):
        part.copy_(torch.empty(part.numel(), device=out.device).normal_(0.0, std, generator=gen).round_()
                   .clamp_(-limit - 1 if limit == 7 else -limit, limit))
    return out


def _weights(gen, shape, kind, scales_per_row):
    """Quantised weights [.., N, K] of a matrix with entries of about 0.02, and their fp32 scales."""
    std, limit = (2.5, 7) if kind == "int4" else (32.0, 127)
    w = _fill(torch.empty(shape, dtype=torch.int8, device="cuda"), gen, std, limit)
    s = torch.rand((*shape[:-1], scales_per_row), generator=gen, device="cuda").add_(0.5).mul_(0.02 / std)
    return w, s


def prepare(case, seed):
    m = MODELS[case["model"]]
    T, H, E, k, I = case["tokens"], m["H"], m["E"], m["k"], m["I"]
    dtype = {"bf16": torch.bfloat16, "fp16": torch.float16}[case["dtype"]]
    int4 = case["weights"] == "int4"
    gen = torch.Generator(device="cuda").manual_seed(seed)
    with torch.device("cuda"):
        # popularity ~ rank^-s over a random order of the experts, as a prior on the logits
        prior = torch.zeros(E)
        if case["zipf"]:
            rank = torch.randperm(E, generator=gen, device="cuda").float() + 1
            prior = -case["zipf"] * rank.log()
        router = AscendFusedTopKRouter(
            k, E, renormalize=True, use_grouped_topk=m["groups"] > 1,
            num_expert_group=m["groups"] if m["groups"] > 1 else None,
            topk_group=m["top_groups"] if m["groups"] > 1 else None, scoring_func=m["scoring"],
            routed_scaling_factor=m["factor"],
            e_score_correction_bias=(torch.randn(E, generator=gen, device="cuda") * 0.01
                                     if m["scoring"] == "sigmoid" else None))
        shared = None
        if case["shared"] != "no":
            (u, us), (d, ds) = _weights(gen, (2 * I, H), "int8", 1), _weights(gen, (H, I), "int8", 1)
            shared = AscendSharedExperts(u, us, d, ds, multistream_overlap=case["shared"] == "side")
        gate = None
        if case["gate"]:
            gate = AscendGateLinear(H, E, bias=bool(case["zipf"]))
            gate.weight.data.normal_(0.0, H ** -0.5, generator=gen)
            if case["zipf"]:
                gate.bias.data.copy_(prior)
        if int4:
            scheme = get_scheme_class("W4A8_DYNAMIC", "moe")(group_size=W4_GROUP, in_dtype=dtype)
        else:
            scheme = get_scheme_class("W8A8_DYNAMIC", "moe")(in_dtype=dtype, dynamic_eplb=case["eplb"])
        layer = AscendRoutedExperts(
            FusedMoEConfig(num_experts=E, experts_per_token=k, hidden_dim=H, intermediate_size_per_partition=I),
            scheme, router, params_dtype=torch.float32, shared_experts=shared, gate=gate, dynamic_eplb=case["eplb"])
        w13, s13 = _weights(gen, (E, 2 * I, H), case["weights"], H // W4_GROUP if int4 else 1)
        w2, s2 = _weights(gen, (E, H, I), case["weights"], I // W4_GROUP if int4 else 1)
        tensors = {"w13_weight": w13, "w13_weight_scale": s13, "w2_weight": w2, "w2_weight_scale": s2}
        if not int4:
            tensors["w13_weight_offset"], tensors["w2_weight_offset"] = torch.zeros_like(s13), torch.zeros_like(s2)
        layer.load_weights(tensors)
        x = torch.randn(T, H, generator=gen, device="cuda").to(dtype)
        logits = None if case["gate"] else torch.randn(T, E, generator=gen, device="cuda") + prior
    return {"layer": layer, "x": x, "logits": logits}


def run(state):
    layer = state["layer"]
    out = layer(state["x"]) if state["logits"] is None else layer(state["x"], state["logits"])
    return out if layer.moe_load is None else {"out": out, "load": layer.moe_load}


def _touched(case):
    """How many experts such a batch touches, by drawing one."""
    m = MODELS[case["model"]]
    T, E, k, groups = case["tokens"], m["E"], m["k"], m["groups"]
    rng = np.random.default_rng(0)
    score = rng.standard_normal((T, E))
    if case["zipf"]:
        score -= case["zipf"] * np.log(rng.permutation(E) + 1.0)
    if groups > 1:
        score = 1.0 / (1.0 + np.exp(-score))
        by_group = score.reshape(T, groups, E // groups)
        best = np.argsort(-np.sort(by_group, axis=2)[:, :, -2:].sum(axis=2), axis=1)[:, m["top_groups"]:]
        np.put_along_axis(by_group, best[:, :, None], -1.0, axis=1)
    return len(np.unique(np.argpartition(-score, k - 1, axis=1)[:, :k]))


def work(case):
    m = MODELS[case["model"]]
    T, H, E, k, I = case["tokens"], m["H"], m["E"], m["k"], m["I"]
    if case["weights"] == "int4":
        expert = 3 * H * I / 2 + 4 * (2 * I * (H // W4_GROUP) + H * (I // W4_GROUP))
    else:
        expert = 3 * H * I + 4 * (2 * I + H)
    nbytes = _touched(case) * expert + 2 * T * H * 2
    flops = 6 * T * k * H * I
    if case["shared"] != "no":
        nbytes += 3 * H * I + 4 * (2 * I + H)
        flops += 6 * T * H * I
    if case["gate"]:
        nbytes += 4 * E * H
        flops += 2 * T * E * H
    else:
        nbytes += 4 * T * E
    if case["eplb"]:
        nbytes += 2 * 8 * E
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # 16-bit outputs of products over int8 activations: a value that another order of the fp32 steps rounds to the
    # neighbouring int8 moves its row by about 1e-2; expert loads are whole numbers, ties of the gate aside
    return {"rel": 1e-2, "max": 0.3, "differ": 2e-3 if case["gate"] else 0.0}
