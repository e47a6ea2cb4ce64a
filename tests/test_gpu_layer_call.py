"""The layer as one native call (``layer(x, logits)``) against the operator-by-operator form
(``layer.forward_impl``): the same bits, over the forms the call chooses between."""
import copy
import dataclasses
import threading

import pytest
import torch

from _inputs import CONFIGS, make_layer
from _layer_utils import build_layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _pair(name, tokens, shape=None, **kw):
    cfg = dataclasses.replace(CONFIGS[name], T=tokens, **(shape or {}))
    d = make_layer(cfg, seed=tokens)
    return cfg, build_layer(cfg, d, DEV, **kw), d["x"].to(DEV), d["logits"].to(DEV)


# one token; the borders of the form for a few tokens (32 pairs, 64 with a shared expert), of pair order (three pairs per expert, 1024
# pairs) and of the one-launch index maps (4096 pairs); a batch with a ragged end on the sorted path
@pytest.mark.parametrize("tokens", [1, 4, 5, 8, 9, 24, 25, 127, 128, 129, 512, 513, 1031])
@pytest.mark.parametrize("name", ["c2_small", "c4_small", "c5_small"])
def test_one_call_equals_the_operators(name, tokens):
    cfg, layer, x, logits = _pair(name, tokens, shared=CONFIGS[name].shared)
    got = layer(x, logits)
    assert layer._layer_plan.desc is not None
    assert torch.equal(got, layer.forward_impl(x, logits).routed_out)


# the form for a few tokens, the shared expert in the pair-order launches (blocks of 32 tokens; a clamp of its own; an
# alpha that only its own operator knows), and the sorted path
@pytest.mark.parametrize("tokens", [1, 8, 32, 33, 64, 96, 127, 300])
@pytest.mark.parametrize("overlap, limit, alpha", [(False, 0.0, 1.0), (True, 0.7, 1.0), (True, 0.7, 1.5)])
def test_shared_expert_in_the_call(tokens, overlap, limit, alpha):
    cfg, layer, x, logits = _pair("c4_small", tokens, shared=True, overlap=overlap)
    layer.shared_experts.swiglu_limit, layer.shared_experts.swiglu_alpha = limit, alpha
    want = layer.forward_impl(x, logits).routed_out
    for _ in range(3):
        assert torch.equal(layer(x, logits), want)


# the shared expert on its own: up to 16 tokens on the kernels for a few tokens (its rows quantised in place, or by a
# launch), beyond that on the dense products
@pytest.mark.parametrize("tokens", [1, 8, 16, 17])
@pytest.mark.parametrize("overlap", [False, True])
@pytest.mark.parametrize("experts", ["sorted int8", "int4"])
def test_shared_expert_beside_the_call(experts, overlap, tokens):
    from vllm_ascend_amd.fused_moe.shared_experts import AscendSharedExperts

    if experts == "int4":
        cfg, layer, x, logits = _pair("c5_small", tokens)
        g = torch.Generator().manual_seed(tokens)
        w = [torch.randint(-127, 128, s, generator=g, dtype=torch.int8).to(DEV) for s in ((2048, cfg.H), (cfg.H, 1024))]
        s = [(torch.rand(n, generator=g) * 0.009 + 0.001).to(DEV) for n in (2048, cfg.H)]
        layer.shared_experts = AscendSharedExperts(w[0], s[0], w[1], s[1], swiglu_limit=0.7, multistream_overlap=overlap)
    else:
        cfg, layer, x, logits = _pair("c4_small", tokens, shared=True, overlap=overlap)
        layer.use_pair_order = False
    want = layer.forward_impl(x, logits).routed_out
    for _ in range(3):
        assert torch.equal(layer(x, logits), want)
    assert layer._layer_plan.desc is not None


@pytest.mark.parametrize("tokens", [2, 4, 60, 300])
def test_weight_lists_and_expert_loads(tokens):
    cfg, layer, x, logits = _pair("c7_small", tokens, dynamic_eplb=True, collect_expert_load=True)
    res = layer.forward_impl(x, logits)
    layer.clear_moe_load()
    assert torch.equal(layer(x, logits), res.routed_out)
    assert torch.equal(layer(x, logits), res.routed_out)
    assert torch.equal(layer.moe_load, 2 * res.expert_tokens)
    layer.w13_weight_list[1] = layer.w13_weight_list[0].clone()  # one expert swapped: the next call sees it
    assert torch.equal(layer(x, logits), layer.forward_impl(x, logits).routed_out)


# the full decode shapes: long K, shared expert with its own arithmetic, rows quantised in place (1 token) or by a launch
@pytest.mark.parametrize("name, tokens", [("c2_qwen3_decode", 1), ("c2_qwen3_decode", 2), ("c6_dsv3_decode", 1),
                                          ("c6_dsv3_decode", 4)])
def test_a_few_tokens_at_full_size(name, tokens):
    cfg = dataclasses.replace(CONFIGS[name], T=tokens)
    d = make_layer(cfg, seed=tokens, gen_device=DEV)
    layer = build_layer(cfg, d, DEV, shared=cfg.shared)
    x = d["x"]
    for shared_args in ((0.0, 1.0, 0.0), (1.5, 1.3, 0.25)):
        if layer.shared_experts is not None:
            layer.shared_experts.swiglu_limit, layer.shared_experts.swiglu_alpha, layer.shared_experts.swiglu_beta = shared_args
        assert torch.equal(layer(x, d["logits"]), layer.forward_impl(x, d["logits"]).routed_out)
    # every token on the same experts, and a row of zeros
    logits = d["logits"][:1].expand(tokens, -1).contiguous()
    x = x.clone()
    x[-1] = 0
    assert torch.equal(layer(x, logits), layer.forward_impl(x, logits).routed_out)


# gating and quantisation inside the first launch: 1 to 4 tokens (130 and 256 experts: one; from two on a launch in front of
# it), experts that fill no register or word of four, groups,
# scores that tie (so the lower index decides) and a row of one score, logits of every type; rows that are no multiple of
# the 512 values a wavefront takes
@pytest.mark.parametrize("tokens", [1, 2, 3, 4])
@pytest.mark.parametrize("experts, k, groups, hidden", [(5, 2, 1, 64), (66, 4, 1, 576), (130, 3, 1, 1088), (256, 4, 8, 512),
                                                        (36, 4, 4, 1024)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_gating_inside_the_first_launch(tokens, experts, k, groups, hidden, dtype):
    shape = dict(E=experts, k=k, H=hidden, I=128, n_group=groups, topk_group=max(1, groups // 2),
                 scoring="sigmoid" if groups > 1 else "softmax", bias=groups > 1)
    cfg, layer, x, logits = _pair("c2_small", tokens, shape)
    flat = logits.clone()
    flat[-1] = 0.25
    for lg in (logits, (logits * 2).round() / 2, flat):
        lg = lg.to(dtype)
        assert torch.equal(layer(x, lg), layer.forward_impl(x, lg).routed_out)
    assert layer._layer_plan.desc is not None


# the router gate's chunk results added up by the launch that gates (up to 16 chunks of 128, the last one whole or half) or
# by a launch of their own (17), with and without a bias, few and many tokens
@pytest.mark.parametrize("tokens", [1, 4, 5, 40, 300])
@pytest.mark.parametrize("hidden, experts", [(64, 8), (960, 66), (1984, 32), (2048, 130), (2112, 32)])
@pytest.mark.parametrize("bias", [False, True])
def test_chunk_results_of_the_gate(tokens, hidden, experts, bias):
    from vllm_ascend_amd.fused_moe.gate_linear import AscendGateLinear

    cfg, layer, x, _ = _pair("c2_small", tokens, dict(H=hidden, E=experts, k=2, I=64))
    layer.gate = AscendGateLinear(hidden, experts, bias=bias, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(tokens)
    layer.gate.weight.data.normal_(0.0, hidden ** -0.5, generator=g)
    if bias:
        layer.gate.bias.data.normal_(0.0, 1.0, generator=g)
    logits, _ = layer.gate(x)
    assert torch.equal(layer(x), layer.forward_impl(x, logits).routed_out)
    assert layer._layer_plan.desc is not None


# pair order with experts of several 32-row blocks (workgroups of their own), the others idle or with a few rows
@pytest.mark.parametrize("tokens", [32, 33, 64, 65, 200])
@pytest.mark.parametrize("rest", [0, 7])
def test_hot_experts_in_pair_order(tokens, rest):
    cfg, layer, x, logits = _pair("c2_small", tokens)
    hot = logits[:1].expand(tokens, -1).contiguous()
    if rest:
        hot[::rest] = logits[::rest]
    assert torch.equal(layer(x, hot), layer.forward_impl(x, hot).routed_out)
    layer.use_fused_small_batch = False
    assert torch.equal(layer(x, hot), layer.forward_impl(x, hot).routed_out)
    want = layer.forward_impl(x, hot).routed_out
    layer.use_fused_small_batch = True
    assert torch.equal(layer(x, hot), want)  # against the operators on the sorted order


# ... with further blocks in front of the slots and no places before them (up to two pairs per expert), and behind them as well;
# an expert of 50 units on both sides of 384 pairs
FURTHER = [(t, dict(E=128, k=4)) for t in (56, 64, 65, 250)] + [(t, dict(I=1600)) for t in (95, 96)]


@pytest.mark.parametrize("tokens, shape", FURTHER)
def test_further_blocks_around_the_slots(tokens, shape):
    cfg, layer, x, logits = _pair("c2_small", tokens, shape)
    hot = logits[:1].expand(tokens, -1).contiguous()
    hot[::5] = logits[::5]
    got = layer(x, hot)
    layer.use_pair_order = False
    assert torch.equal(got, layer(x, hot))


# few experts: the last batch in pair order, and the first whose experts would read 128 MiB again (or have 36 rows each), by
# the operators' line; with a shared expert in the same launches the layer's lies at 256 MiB, which neither reaches
@pytest.mark.parametrize("shape, tokens", [(dict(E=8, k=2, H=1024, I=1408), 497), (dict(E=16, k=2, H=2048, I=1408), 288)])
@pytest.mark.parametrize("shared", [False, True])
def test_few_experts_with_many_rows_are_sorted(shape, tokens, shared):
    from vllm_ascend_amd import kernels as K

    for T, pair_order in ((tokens - 1, True), (tokens, False)):
        print(f"{shape} {T} tokens shared={shared}", flush=True)
        assert K.pair_order(T, shape["k"], shape["E"], shape["E"], shape["H"], shape["I"]) is pair_order
        cfg, layer, x, logits = _pair("c2_small", T, dict(shape, shared=shared), shared=shared)
        assert (layer.shared_experts is not None) == shared
        got = layer(x, logits)
        assert torch.equal(got, layer.forward_impl(x, logits).routed_out)
        layer.use_pair_order = False
        assert torch.equal(got, layer(x, logits))
        assert torch.equal(got, layer.forward_impl(x, logits).routed_out)


# ... the last batch in pair order with a shared expert in the launches, and the first one without
@pytest.mark.parametrize("overlap", [False, True])
def test_few_experts_with_a_shared_expert_are_sorted_later(overlap):
    shape = dict(E=8, k=2, H=4096, I=2048)
    for T in (170, 171):
        cfg, layer, x, logits = _pair("c2_small", T, dict(shape, shared=True), shared=True, overlap=overlap)
        assert layer.shared_experts is not None
        got = layer(x, logits)
        assert torch.equal(got, layer.forward_impl(x, logits).routed_out)
        layer.use_pair_order = False
        assert torch.equal(got, layer(x, logits))


# a shared expert in the launches of a layer whose down product could re-quantise inside
@pytest.mark.parametrize("tokens", [9, 57, 127])
@pytest.mark.parametrize("overlap", [False, True])
def test_shared_expert_instead_of_the_re_quantisation(tokens, overlap):
    shape = dict(E=128, k=8, H=1024, I=320, shared=True)
    cfg, layer, x, logits = _pair("c2_small", tokens, shape, shared=True, overlap=overlap)
    assert layer.shared_experts is not None
    assert torch.equal(layer(x, logits), layer.forward_impl(x, logits).routed_out)
    assert layer._layer_plan.desc is not None


# int4 weights in pair order (up to 40 tokens of experts this small): one block of 16 or 32 rows and several, one scale per channel or per group, hot and idle experts
@pytest.mark.parametrize("tokens", [1, 16, 17, 32, 33, 40, 41])
@pytest.mark.parametrize("name", ["c5_small", "c5_small_perchannel"])
def test_int4_pair_order(name, tokens):
    cfg, layer, x, logits = _pair(name, tokens)
    hot = logits[:1].expand(tokens, -1).contiguous()
    hot[::9] = logits[::9]
    for lg in (logits, hot):
        assert torch.equal(layer(x, lg), layer.forward_impl(x, lg).routed_out)


# the same: fewer K blocks than the ring holds, no multiple of it, channels that leave wavefronts of a workgroup idle; an
# expert named more than once by a token (more rows than tokens: further passes over its weights)
@pytest.mark.parametrize("H,I,tokens", [(64, 64, 1), (192, 64, 16), (448, 320, 17), (832, 448, 32)])
def test_int4_pair_order_edges(H, I, tokens):
    cfg, layer, x, logits = _pair("c5_small_perchannel", tokens, dict(H=H, I=I))
    assert torch.equal(layer(x, logits), layer.forward_impl(x, logits).routed_out)
    select = layer.router.select_experts

    def repeated(*a, **kw):
        weights, ids = select(*a, **kw)
        ids = ids.clone()
        ids[:, 1:3] = 3
        return weights, ids

    layer.router.select_experts = repeated
    weights, ids = repeated(x, logits)
    want = layer.quant_method.apply(layer, x, weights, ids, None, None).routed_out
    assert torch.equal(layer(x, logits), want)


def test_the_call_follows_the_layer():
    """Options that change between calls, and a copied layer."""
    cfg, layer, x, logits = _pair("c2_small", 40)
    layer(x, logits)
    for change in (dict(use_pair_order=False), dict(use_fused_small_batch=False), dict(use_fused_small_batch=True)):
        for k, v in change.items():
            setattr(layer, k, v)
        assert torch.equal(layer(x, logits), layer.forward_impl(x, logits).routed_out)
    layer.router.renormalize = not layer.router.renormalize
    assert torch.equal(layer(x, logits), layer.forward_impl(x, logits).routed_out)
    half = logits.to(torch.bfloat16)
    assert torch.equal(layer(x, half), layer.forward_impl(x, half).routed_out)
    assert torch.equal(layer(x[::2], logits[::2]), layer.forward_impl(x[::2], logits[::2]).routed_out)
    twin = copy.deepcopy(layer)
    assert torch.equal(twin(x, logits), layer.forward_impl(x, logits).routed_out)


@pytest.mark.parametrize("name", ["c2_small", "c5_small"])
def test_a_router_with_a_selection_of_its_own(name):
    """Its ids are the ones the experts run on, through the call and through the operators."""
    cfg, layer, x, logits = _pair(name, 40)
    stock = layer(x, logits)
    select, seen = layer.router.select_experts, []

    def shifted(*a, **kw):
        weights, ids = select(*a, **kw)
        seen.append(1)
        return weights, ((ids + 1) % cfg.E).to(torch.int32)

    layer.router.select_experts = shifted
    weights, ids = shifted(x, logits)
    want = layer.quant_method.apply(layer, x, weights, ids, None, None).routed_out
    assert torch.equal(layer(x, logits), want) and torch.equal(layer.forward_impl(x, logits).routed_out, want)
    assert len(seen) == 3 and not torch.equal(want, stock)


# one layer, several calls at a time: sorted batches small enough for one routing workgroup, pair order, the kernels for
# a few tokens, the shared expert on its side stream
AT_A_TIME = [("c5_small", 60, {}, {}), ("c2_small", 48, {}, dict(use_pair_order=False)), ("c2_small", 48, {}, {}),
             ("c4_small", 8, dict(shared=True, overlap=True), {}),
             ("c4_small", 300, dict(shared=True, overlap=True), {}),
             ("c4_small", 96, dict(shared=True, overlap=True), dict(use_pair_order=False))]


def _two_batches(name, tokens, kw, options):
    cfg, layer, x, logits = _pair(name, tokens, **kw)
    for k, v in options.items():
        setattr(layer, k, v)
    batches = [(x, logits), (x.flip(0).contiguous(), logits.roll(1, 1).contiguous()[: tokens - 1])]
    batches[1] = (batches[1][0][: tokens - 1], batches[1][1])
    return layer, batches, [layer.forward_impl(*b).routed_out for b in batches]


@pytest.mark.parametrize("name, tokens, kw, options", AT_A_TIME)
def test_one_layer_on_two_streams(name, tokens, kw, options):
    print(f"two streams: {name} {tokens} {kw} {options}", flush=True)
    layer, batches, want = _two_batches(name, tokens, kw, options)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(20):
        for s, b, out in zip(streams, batches, got):
            with torch.cuda.stream(s):
                out.append(layer(*b))
    torch.cuda.synchronize()
    for out, w in zip(got, want):
        assert all(torch.equal(o, w) for o in out)


@pytest.mark.parametrize("whole", [True, False])
@pytest.mark.parametrize("name, tokens, kw, options", AT_A_TIME)
def test_one_layer_on_two_threads(name, tokens, kw, options, whole):
    print(f"two threads: {name} {tokens} {kw} {options} whole={whole}", flush=True)
    layer, batches, want = _two_batches(name, tokens, kw, options)
    torch.cuda.synchronize()
    got, failed = [[], []], []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    got[i].append(layer(*batches[i]) if whole else layer.forward_impl(*batches[i]).routed_out)
                torch.cuda.current_stream().synchronize()
        except Exception as exc:  # noqa: BLE001 -- reported by the test's own thread
            failed.append(exc)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed
    for out, w in zip(got, want):
        assert len(out) == 20 and all(torch.equal(o, w) for o in out)


@pytest.mark.parametrize("name", ["c5_small", "c2_small"])
def test_gating_sort_and_quantisation_in_one_launch(name):
    """The form of a caller of the library that runs the layer on one stream and brings the counter."""
    cfg, layer, x, logits = _pair(name, 60)
    layer.use_pair_order = False
    want = layer(x, logits)
    counter = torch.zeros(1, dtype=torch.int32, device=DEV)
    plan = layer._layer_plan
    plan.desc.sync_counter = counter.data_ptr()
    plan.sizes.clear()
    for _ in range(3):
        assert torch.equal(layer(x, logits), want)
    assert layer._layer_plan is plan and int(counter) == 0


# pair order, the sorted path, and a few tokens: the combine counts the pairs of every expert only where loads are kept
@pytest.mark.parametrize("tokens", [2, 48, 300])
def test_expert_loads_without_weight_lists(tokens):
    cfg, layer, x, logits = _pair("c2_small", tokens, collect_expert_load=True)
    res = layer.forward_impl(x, logits)
    layer.clear_moe_load()
    for n in (1, 2):
        assert torch.equal(layer(x, logits), res.routed_out)
        assert torch.equal(layer.moe_load, n * res.expert_tokens)
    layer.eplb_heat_collection_status = False
    assert torch.equal(layer(x, logits), res.routed_out)
    assert torch.equal(layer.moe_load, 2 * res.expert_tokens)


@pytest.mark.parametrize("name, tokens, kw", [("c2_small", 2, {}), ("c2_small", 48, {}), ("c2_small", 300, {}),
                                              ("c4_small", 96, dict(shared=True)), ("c4_small", 300, dict(shared=True)),
                                              ("c5_small", 16, {}), ("c5_small", 80, {})])
def test_measurement_hook_brackets_the_routed_gate_up_product(name, tokens, kw):
    import ctypes

    from vllm_ascend_amd._lib import load

    cfg, layer, x, logits = _pair(name, tokens, **kw)
    want = layer(x, logits)
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    buf = torch.zeros(2, 1 << 28, dtype=torch.int32, device=DEV)

    def around_copies():  # an interval (milliseconds) that the bracketed kernel cannot have
        ev0.record()
        for _ in range(8):
            buf[1].copy_(buf[0])
        ev1.record()
        torch.cuda.synchronize()
        return ev0.elapsed_time(ev1)

    before = around_copies()  # creates the handles
    load().moe355_profile_next_gemm(ctypes.c_void_p(ev0.cuda_event), ctypes.c_void_p(ev1.cuda_event))
    assert torch.equal(layer(x, logits), want)
    torch.cuda.synchronize()
    first = ev0.elapsed_time(ev1)
    print(f"hook {name} {tokens}: {before * 1e3:.1f} -> {first * 1e3:.1f} us", flush=True)
    assert before > 1.0 and 5e-4 < first < before / 2
    again = around_copies()
    layer(x, logits)  # the events were taken by the call before
    torch.cuda.synchronize()
    assert ev0.elapsed_time(ev1) == again > before / 2


# every form of the call: a few tokens (their rows quantised in place; by a launch; with the shared expert), pair order
# (a launch re-quantises; the down GEMM does, rows of one and of several loads; the shared expert in the launches), int4
# in pair order and sorted, the sorted path with the shared expert in line and on its side stream, per-expert weight
# tables
_REQ = dict(H=1024, E=128, k=8)
FORMS = [("c2_small", 2, {}), ("c2_small", 2, dict(shape=dict(H=1024, E=128, k=8, I=1408))),
         ("c4_small", 2, dict(shared=True)), ("c2_small", 24, {}), ("c2_small", 100, {}),
         ("c2_small", 40, dict(shape=dict(I=320, **_REQ))), ("c2_small", 40, dict(shape=dict(I=1408, **_REQ))),
         ("c4_small", 40, dict(shared=True)), ("c4_small", 96, dict(shared=True, overlap=True)), ("c5_small", 12, {}),
         ("c5_small", 80, {}), ("c4_small", 300, dict(shared=True)), ("c4_small", 300, dict(shared=True, overlap=True)),
         ("c7_small", 40, dict(dynamic_eplb=True)), ("c7_small", 300, dict(dynamic_eplb=True))]


def _as_fp16(layer, x):
    layer.quant_method.in_dtype = torch.float16
    return x.to(torch.float16)


@pytest.mark.parametrize("name, tokens, kw", FORMS)
@pytest.mark.parametrize("gate", [False, True])
def test_a_captured_call_replays_on_new_inputs(name, tokens, kw, gate):
    """Replays with other inputs in the captured buffers, eager work and synchronisations between them."""
    from vllm_ascend_amd.fused_moe.gate_linear import AscendGateLinear

    print(f"capture {name} {tokens} {kw} gate={gate}", flush=True)
    cfg, layer, x, logits = _pair(name, tokens, **kw)
    if gate:
        layer.gate = AscendGateLinear(cfg.H, cfg.E, device=DEV)
        layer.gate.weight.data.normal_(0.0, cfg.H ** -0.5)
    args = (x,) if gate else (x, logits)
    for _ in range(2):
        layer(*args)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer(*args)
    first = [a.clone() for a in args]
    for shift in (0, 1, 5, 0):
        for a, f in zip(args, first):
            a.copy_(f.roll(shift, 0) * (1.0 + shift))
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        assert torch.equal(got, layer(*args))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, got)


@pytest.mark.parametrize("name, tokens, kw", FORMS)
def test_fp16_hidden_states_in_the_call(name, tokens, kw):
    cfg, layer, x, logits = _pair(name, tokens, **kw)
    x = _as_fp16(layer, x)
    got = layer(x, logits)
    assert got.dtype == torch.float16 and layer._layer_plan.desc is not None
    assert torch.equal(got, layer.forward_impl(x, logits).routed_out)
    layer.use_fused_small_batch = False
    assert torch.equal(got, layer.forward_impl(x, logits).routed_out)


def _same_values(a, b):
    return bool((((a == b) | (a.isnan() & b.isnan()))).all())


# an infinity or a NaN in a token's hidden states (the row's maximum, and through the scale its SwiGLU values), a value
# large enough for the products to overflow: the operators on the sorted order say what comes out, and the other tokens'
# rows must not notice
@pytest.mark.parametrize("name, tokens, kw", FORMS)
def test_infinities_and_nans(name, tokens, kw):
    print(f"inf and nan {name} {tokens} {kw}", flush=True)
    cfg, layer, x, logits = _pair(name, tokens, **kw)
    if "shape" in kw and tokens > 2:
        from vllm_ascend_amd.kernels import gmm2_requant_pairs_supported

        assert gmm2_requant_pairs_supported(tokens, cfg.k, cfg.H, cfg.I, cfg.E)
    clean = layer(x, logits)
    rows = {0: float("inf"), tokens // 2: float("nan"), tokens - 1: -3e38}
    for t, v in rows.items():
        x[t, 7 * t % cfg.H] = v
    got = layer(x, logits)
    layer.use_fused_small_batch = False
    want = layer.forward_impl(x, logits).routed_out
    layer.use_fused_small_batch = True
    assert _same_values(got, want) and _same_values(layer.forward_impl(x, logits).routed_out, want)
    others = [t for t in range(tokens) if t not in rows]
    assert torch.equal(got[others], clean[others])


# scales that start in the middle of a 16-byte line: what the operators refuse, the call refuses in each of its forms
@pytest.mark.parametrize("name, tokens, kw, where", [
    ("c2_small", 2, {}, "w13_weight_scale_fp32"), ("c2_small", 2, {}, "w2_weight_scale_fp32"),
    ("c2_small", 48, {}, "w13_weight_scale_fp32"), ("c2_small", 300, {}, "w2_weight_scale_fp32"),
    ("c5_small", 12, {}, "w13_weight_scale"), ("c5_small", 12, {}, "w2_weight_scale"),
    ("c5_small", 80, {}, "w2_weight_scale"),
    ("c4_small", 2, dict(shared=True), "down_scale_fp32"), ("c4_small", 96, dict(shared=True), "down_scale_fp32"),
    ("c4_small", 300, dict(shared=True), "down_scale_fp32")])
def test_misaligned_scales_are_refused(name, tokens, kw, where):
    from vllm_ascend_amd._lib import Moe355Error

    cfg, layer, x, logits = _pair(name, tokens, **kw)
    layer(x, logits)
    owner = layer.shared_experts if where == "down_scale_fp32" else layer
    t = getattr(owner, where)
    shifted = torch.empty(t.numel() + 1, device=DEV)[1:].view(t.shape)
    shifted.copy_(t)
    if isinstance(t, torch.nn.Parameter):
        t.data = shifted
    else:
        setattr(owner, where, shifted)
    with pytest.raises(Moe355Error, match="alignment"):
        layer.forward_impl(x, logits)
    with pytest.raises(Moe355Error, match="alignment"):
        layer(x, logits)
