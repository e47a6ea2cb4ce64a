"""The layer as one native call (``moe355_layer_forward``): the same operators, chosen by the same rules, as
``AscendRoutedExperts.forward_impl`` (``vllm_ascend/ops/fused_moe/routed_experts.py:496-609``) enqueues one by one, so
the output is the same, bit for bit.

A decode step of a small layer is bound by the host: going operator by operator costs 50 to 240 us of interpreter,
allocations and event records for 27 to 200 us of kernels.  Here a call is two allocations and one foreign call; what
the library needs to know about the layer is gathered once and kept until something about the layer changes."""
from __future__ import annotations

import ctypes
from operator import itemgetter

import torch
from torch.nn.modules.module import _global_forward_hooks, _global_forward_pre_hooks

from .. import _lib
from ..kernels import _DT, _stream
from ..quantization.w4a8 import AscendW4A8DynamicFusedMoEMethod
from ..quantization.w8a8_dynamic import AscendW8A8DynamicFusedMoEMethod
from .gate_linear import AscendGateLinear
from .moe_comm_method import AllGatherCommImpl, _IdentityPrepareFinalize
from .router import AscendFusedTopKRouter
from .shared_experts import AscendSharedExperts, shared_experts_calculation_stream

_MAX_SIZES = 256  # batch sizes whose scratch size is remembered
_INT8, _INT8_LIST, _INT4 = 0, 1, 2  # moe355_layer.weights


class _Plan:
    """What one layer looks like to the library; ``desc`` is None when the native call cannot take it."""

    __slots__ = ("key", "desc", "ref", "hidden", "experts", "sizes", "bias", "forward", "workspace")

    def __init__(self, key):
        self.key = key
        self.desc = self.ref = None
        self.sizes = {}

    def __reduce__(self):  # a copied or pickled layer makes its own
        return type(None), ()


def _view(t):
    """What the library is told of a tensor (its address) and what that address stands for.  All of it is compared on
    every call and nothing keeps a tensor alive: an address alone may belong to another tensor of another type or size
    by the time of the next call."""
    return t.data_ptr(), t.dtype, t.shape, t.is_contiguous(), t.get_device()


def _is(view, dtype, shape, device):
    return view[1:] == (dtype, shape, True, device)


def _holds(view, dtype, numel, device):
    return view[1] == dtype and view[2].numel() == numel and view[3:] == (True, device)


# what of a layer, its router and its shared expert a plan is made from
_LAYER = itemgetter("quant_method", "router", "moe_config", "moe_comm_method", "activation",
                    "apply_router_weight_on_input", "ascend_expert_map", "global_redundant_expert_num",
                    "ascend_mc2_mask", "ascend_pertoken_scale", "enable_force_load_balance", "log2phy",
                    "use_fused_small_batch", "use_pair_order", "dynamic_eplb", "eplb_heat_collection_status",
                    "multi_stage")
_ROUTER = itemgetter("top_k", "renormalize", "num_expert_group", "topk_group", "scoring_func",
                     "routed_scaling_factor", "e_score_correction_bias")
_SHARED = itemgetter("multistream_overlap", "swiglu_limit", "swiglu_alpha", "swiglu_beta", "gate_up_weight",
                     "down_weight", "gate_up_scale_fp32", "down_scale_fp32", "_forward_hooks", "_forward_pre_hooks")
# what a call runs when nothing has been put in its place, in a subclass, on an instance or in the class itself
_SELECT_EXPERTS, _GUARD = AscendFusedTopKRouter.select_experts, AscendFusedTopKRouter.is_fused_supported
_SHARED_FORWARD, _GATE_FORWARD = AscendSharedExperts.forward, AscendGateLinear.forward
_INT8_APPLY = AscendW8A8DynamicFusedMoEMethod.apply_small_batch
_INT4_APPLY = AscendW4A8DynamicFusedMoEMethod.apply_small_batch
_INT8_SCALES = itemgetter("w13_weight_scale_fp32", "w2_weight_scale_fp32")
_INT4_TENSORS = itemgetter("w13_weight", "w13_weight_scale", "w2_weight", "w2_weight_scale")
_LISTS = itemgetter("w13_weight_list", "w13_weight_scale_fp32_list", "w2_weight_list", "w2_weight_scale_list")


def _key(layer, x_dtype, device, logits_dtype):
    """Everything that the plan of such a call is made from, or None where the call goes operator by operator: an
    option or a part that the library has no whole form for, or a layer that is not put together as
    ``AscendRoutedExperts.__init__`` and the two schemes do it (another scheme, router or shared expert, a gate that is
    any callable, a tensor registered under the name of an attribute), or one with a method or hook of the caller's in
    it.  Compared on every call, so plain dictionary lookups: types first, then what such types have."""
    d = layer.__dict__
    try:
        (q, r, cfg, comm, act, on_input, expert_map, redundant, mc2_mask, pertoken, forced, log2phy, fused, pair_order,
         eplb, collecting, staged) = _LAYER(d)
        if (on_input or expert_map is not None or redundant or mc2_mask is not None or pertoken is not None or forced
                or log2phy is not None or not fused):
            return None
        if act != "silu" and (getattr(act, "value", act) or "silu") != "silu":
            return None
        if type(r) is not AscendFusedTopKRouter or type(comm) is not AllGatherCommImpl \
                or type(comm.prepare_finalize) is not _IdentityPrepareFinalize:
            return None
        rd, qd, cd = r.__dict__, q.__dict__, comm.__dict__
        if (AscendFusedTopKRouter.select_experts is not _SELECT_EXPERTS or "select_experts" in rd
                or "_compute_routing" in rd or AscendFusedTopKRouter.is_fused_supported is not _GUARD
                or "is_fused_supported" in rd or "apply_small_batch" in qd or "supports_small_batch" in qd
                or "apply" in qd or "prepare" in cd or "finalize" in cd or "fused_experts" in cd
                or comm.prepare_finalize.__dict__):
            return None
        p = d["_parameters"]
        if type(q) is AscendW8A8DynamicFusedMoEMethod:
            if AscendW8A8DynamicFusedMoEMethod.apply_small_batch is not _INT8_APPLY:
                return None
            if q.use_expert_weight_list:
                weights, w = _INT8_LIST, tuple((len(t), t.table.data_ptr(), _view(t[0])) for t in _LISTS(d))
            else:
                s13, s2 = _INT8_SCALES(d)
                weights = _INT8
                w = (_view(p["w13_weight"]), _view(s13), _view(p["w2_weight"]), _view(s2))
        elif type(q) is AscendW4A8DynamicFusedMoEMethod and not q.use_expert_weight_list:
            if AscendW4A8DynamicFusedMoEMethod.apply_small_batch is not _INT4_APPLY:
                return None
            weights, w = _INT4, tuple(_view(t) for t in _INT4_TENSORS(p))
        else:
            return None
        if q.in_dtype != x_dtype:
            return None
        routing = _ROUTER(rd)
        bias = routing[6]
        m = d["_modules"]
        shared = m["shared_experts"] if "shared_experts" in m else d["shared_experts"]
        sh = g = load = None
        if shared is not None:
            if type(shared) is not AscendSharedExperts:
                return None
            s = shared.__dict__
            sh = _SHARED(s)
            if (AscendSharedExperts.forward is not _SHARED_FORWARD or "forward" in s or "_mlp" in s or "wait" in s
                    or sh[8] or sh[9] or _global_forward_hooks or _global_forward_pre_hooks):
                return None
            sh = (*sh[:4], _view(sh[4]), _view(sh[5]), _view(sh[6]), _view(sh[7]))
        if logits_dtype is None:
            gate = m["gate"] if "gate" in m else d["gate"]
            if type(gate) is not AscendGateLinear:
                return None
            s = gate.__dict__
            if (AscendGateLinear.forward is not _GATE_FORWARD or "forward" in s or s["_forward_hooks"]
                    or s["_forward_pre_hooks"] or _global_forward_hooks or _global_forward_pre_hooks):
                return None
            gp = s["_parameters"]
            gate_bias = gp["bias"] if "bias" in gp else s["bias"]
            g = (_view(gp["weight"]), None if gate_bias is None else _view(gate_bias))
        if eplb and collecting:
            if staged:
                return None  # one row of loads per pass, indexed on the device
            load = _view(d["_buffers"]["moe_load"])
        return (x_dtype, device, logits_dtype, weights, w, sh, g, routing[:6], None if bias is None else _view(bias),
                pair_order, load, cfg.num_experts, cfg.hidden_dim, cfg.intermediate_size_per_partition,
                cfg.swiglu_limit)
    except (AttributeError, KeyError):
        return None


def _make_plan(layer, x, logits, key) -> _Plan:
    """What the key says, as the library takes it; no description where a tensor is not what the library would read
    (weights that have not been laid out, a scale of another type, a tensor elsewhere): the operators convert it or say
    what is wrong with it."""
    logits_dtype = torch.float32 if logits is None else logits.dtype
    r = layer.router
    plan = _Plan(key)
    if x.dtype not in (torch.bfloat16, torch.float16) or not r.is_fused_supported(x):
        return plan
    bias = r.e_score_correction_bias
    if bias is not None and bias.dtype != logits_dtype:
        bias = r.e_score_correction_bias = bias.to(logits_dtype)
        key = plan.key = _key(layer, x.dtype, x.get_device(), None if logits is None else logits_dtype)
        if key is None:
            return plan
    # another thread's call with logits of another type may replace the converted bias while this call uses it
    plan.bias = bias
    (_, dev, _, weights, w, sh, g, routing, bias_view, pair_order, load, E, H, I, limit) = key
    if bias_view is not None and not _is(bias_view, logits_dtype, (E,), dev):
        return plan
    if weights == _INT8_LIST:
        if any(n != E for n, _, _ in w):
            return plan
        addresses, (w13, s13, w2, s2) = [table for _, table, _ in w], [first for _, _, first in w]
        if not (_is(w13, torch.int8, (H, 2 * I), dev) and _holds(s13, torch.float32, 2 * I, dev)
                and _is(w2, torch.int8, (I, H), dev) and _holds(s2, torch.float32, H, dev)):
            return plan
    else:
        addresses, (w13, s13, w2, s2) = [view[0] for view in w], w
        if weights == _INT8:
            if not (_is(w13, torch.int8, (E, H, 2 * I), dev) and _holds(s13, torch.float32, E * 2 * I, dev)
                    and _is(w2, torch.int8, (E, I, H), dev) and _holds(s2, torch.float32, E * H, dev)):
                return plan
        else:
            if len(s13[2]) != 3 or len(s2[2]) != 3:
                return plan
            G13, G2 = s13[2][1], s2[2][1]
            if not (_holds(w13, torch.uint8, E * I * H, dev) and _is(s13, torch.float32, (E, G13, 2 * I), dev)
                    and _holds(w2, torch.uint8, E * H * I // 2, dev) and _is(s2, torch.float32, (E, G2, H), dev)):
                return plan
    lib = _lib.load()
    a = _lib.Layer()
    a.hidden, a.intermediate, a.num_experts = H, I, E
    a.top_k, renormalize, group_count, k_group, scoring_func, a.routed_scaling_factor = routing
    a.k_group = k_group if k_group is not None else 1
    a.group_count = group_count if group_count is not None else 1
    a.renorm, a.norm_type = int(renormalize), 0 if scoring_func == "softmax" else 1
    a.eps, a.swiglu_limit = 1e-20, limit or 0.0
    a.x_dtype, a.bias = _DT[x.dtype], None if bias_view is None else bias_view[0]
    a.weights = weights
    a.w13, a.s13, a.w2, a.s2 = addresses
    if weights == _INT4:
        a.group13, a.group2 = H // G13, I // G2
    # no sync_counter: one counter would be shared by all the streams, threads and graphs that run the layer
    a.pair_order = int(pair_order)
    if g is not None:
        weight, gate_bias = g
        if not _is(weight, torch.float32, (E, H), dev):
            return plan
        if gate_bias is not None and not _holds(gate_bias, torch.float32, E, dev):
            return plan
        a.gate_weight, a.gate_bias = weight[0], None if gate_bias is None else gate_bias[0]
    if sh is not None:
        overlap, a.shared_limit, a.shared_alpha, a.shared_beta, up, down, up_scale, down_scale = sh
        n = up[2][1] if len(up[2]) == 2 else 1
        if n % 2 or not (_is(up, torch.int8, (H, n), dev) and _is(down, torch.int8, (n // 2, H), dev)
                         and _holds(up_scale, torch.float32, n, dev) and _holds(down_scale, torch.float32, H, dev)):
            return plan
        a.shared_intermediate = n // 2
        a.shared = 2 if overlap else 1
        a.shared_w13, a.shared_s13, a.shared_w2, a.shared_s2 = up[0], up_scale[0], down[0], down_scale[0]
        if overlap:
            a.shared_stream = shared_experts_calculation_stream(dev).cuda_stream
    if load is not None:
        if not _is(load, torch.int64, (E,), dev):
            return plan
        a.load = load[0]
    plan.desc, plan.ref = a, ctypes.addressof(a)
    plan.hidden, plan.experts = H, E
    plan.forward, plan.workspace = lib.moe355_layer_forward, lib.moe355_layer_workspace
    return plan


def layer_call(layer, x: torch.Tensor, logits: torch.Tensor | None) -> torch.Tensor | None:
    """The layer's output, or None when the call has to go operator by operator (an option the library has no whole
    form for, or arguments that the operators refuse with a message of their own)."""
    device = x.get_device()
    key = _key(layer, x.dtype, device, None if logits is None else logits.dtype)
    shape = x.shape
    if key is None or not x.is_cuda or len(shape) != 2:
        return None
    d = layer.__dict__
    plan = d.get("_layer_plan")
    if plan is None or plan.key != key:
        if shape[1] != layer.moe_config.hidden_dim or (logits is not None and logits.dtype not in _DT):
            return None
        plan = d["_layer_plan"] = _make_plan(layer, x, logits, key)
    if plan.desc is None:
        return None
    if shape[1] != plan.hidden or not x.is_contiguous():
        return None
    T = shape[0]
    if T == 0:
        return None
    if logits is not None:
        if logits.shape != (T, plan.experts) or not logits.is_contiguous() or logits.get_device() != device:
            return None
        logits_ptr, logits_dtype = logits.data_ptr(), _DT[logits.dtype]
    else:
        logits_ptr, logits_dtype = None, 0
    nbytes = plan.sizes.get(T)
    if nbytes is None:
        if len(plan.sizes) >= _MAX_SIZES:
            plan.sizes.clear()
        nbytes = plan.sizes[T] = plan.workspace(plan.ref, T)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    out = torch.empty_like(x)
    if plan.forward(plan.ref, x.data_ptr(), logits_ptr, logits_dtype, T, out.data_ptr(), ws.data_ptr(), nbytes,
                    _stream(x)):
        return None  # refused before its first launch or in between: nothing of it is visible to the caller
    return out
