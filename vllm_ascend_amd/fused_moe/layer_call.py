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
_WEIGHTS = 2  # ... and where a key holds it


class _Plan:
    """What one layer looks like to the library; ``desc`` is None when the native call cannot take it."""

    __slots__ = ("key", "desc", "ref", "hidden", "experts", "sizes", "forward", "workspace")

    def __init__(self, key):
        self.key = key
        self.desc = self.ref = None
        self.sizes = {}

    def __reduce__(self):  # a copied or pickled layer makes its own
        return type(None), ()


def _ptr(t):
    return None if t is None else t.data_ptr()


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
_INT8_SCALES = itemgetter("w13_weight_scale_fp32", "w2_weight_scale_fp32")
_INT4_TENSORS = itemgetter("w13_weight", "w2_weight", "w13_weight_scale", "w2_weight_scale")
_LISTS = itemgetter("w13_weight_list", "w13_weight_scale_fp32_list", "w2_weight_list", "w2_weight_scale_list")


def _key(layer, x_dtype, logits_dtype):
    """Everything that the plan of such a call is made from, or None where the call goes operator by operator: an
    option or a part that the library has no whole form for, or a layer that is not put together as
    ``AscendRoutedExperts.__init__`` and the two schemes do it (another scheme, router or shared expert, a gate that is
    any callable, a tensor registered under the name of an attribute).  Compared on every call, so plain dictionary
    lookups: types first, then what such types have."""
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
        p = d["_parameters"]
        if type(q) is AscendW8A8DynamicFusedMoEMethod:
            if q.use_expert_weight_list:
                weights, w = _INT8_LIST, tuple(t.table.data_ptr() for t in _LISTS(d))
            else:
                s13, s2 = _INT8_SCALES(d)
                weights = _INT8
                w = (p["w13_weight"].data_ptr(), p["w2_weight"].data_ptr(), s13.data_ptr(), s2.data_ptr())
        elif type(q) is AscendW4A8DynamicFusedMoEMethod and not q.use_expert_weight_list:
            weights, w = _INT4, tuple(t.data_ptr() for t in _INT4_TENSORS(p))
        else:
            return None
        if q.in_dtype != x_dtype:
            return None
        routing = _ROUTER(r.__dict__)
        bias = routing[6]
        m = d["_modules"]
        shared = m["shared_experts"] if "shared_experts" in m else d["shared_experts"]
        sh = g = load = None
        if shared is not None:
            if type(shared) is not AscendSharedExperts:
                return None
            sh = _SHARED(shared.__dict__)
            if sh[8] or sh[9]:
                return None  # hooks
            sh = (*sh[:4], sh[4].data_ptr(), sh[5].data_ptr(), sh[6].data_ptr(), sh[7].data_ptr())
        if logits_dtype is None:
            gate = m["gate"] if "gate" in m else d["gate"]
            if type(gate) is not AscendGateLinear:
                return None
            s = gate.__dict__
            if s["_forward_hooks"] or s["_forward_pre_hooks"]:
                return None
            gp = s["_parameters"]
            gate_bias = gp["bias"] if "bias" in gp else s["bias"]
            g = (gp["weight"].data_ptr(), None if gate_bias is None else gate_bias.data_ptr())
        if eplb and collecting:
            if staged:
                return None  # one row of loads per pass, indexed on the device
            load = d["_buffers"]["moe_load"].data_ptr()
        return (x_dtype, logits_dtype, weights, w, sh, g, routing[:6], None if bias is None else bias.data_ptr(), pair_order,
                load, cfg.num_experts, cfg.hidden_dim, cfg.intermediate_size_per_partition, cfg.swiglu_limit)
    except (AttributeError, KeyError):
        return None


def _make_plan(layer, x, logits, key) -> _Plan:
    logits_dtype = torch.float32 if logits is None else logits.dtype
    r, gate, shared, cfg = layer.router, layer.gate, layer.shared_experts, layer.moe_config
    plan = _Plan(key)
    if x.dtype not in (torch.bfloat16, torch.float16) or not r.is_fused_supported(x):
        return plan
    bias = r.e_score_correction_bias
    if bias is not None:
        if bias.dtype != logits_dtype:
            bias = r.e_score_correction_bias = bias.to(logits_dtype)
            plan.key = _key(layer, x.dtype, None if logits is None else logits_dtype)
        if bias.dim() != 1 or bias.numel() != cfg.num_experts or not bias.is_contiguous() or not bias.is_cuda:
            return plan
    lib = _lib.load()
    E, I = cfg.num_experts, cfg.intermediate_size_per_partition
    a = _lib.Layer()
    a.hidden, a.intermediate, a.num_experts, a.top_k = cfg.hidden_dim, I, E, r.top_k
    a.k_group = r.topk_group if r.topk_group is not None else 1
    a.group_count = r.num_expert_group if r.num_expert_group is not None else 1
    a.renorm, a.norm_type = int(r.renormalize), 0 if r.scoring_func == "softmax" else 1
    a.routed_scaling_factor, a.eps, a.swiglu_limit = r.routed_scaling_factor, 1e-20, cfg.swiglu_limit or 0.0
    a.x_dtype, a.bias = _DT[x.dtype], _ptr(bias)
    a.weights = key[_WEIGHTS]
    if a.weights == _INT8_LIST:
        lists = (layer.w13_weight_list, layer.w13_weight_scale_fp32_list, layer.w2_weight_list,
                 layer.w2_weight_scale_list)
        a.w13, a.s13, a.w2, a.s2 = (t.table.data_ptr() for t in lists)
        sizes = [(t[0].numel() * len(t), t[0].dtype) for t in lists]
    elif a.weights == _INT4:
        s13, s2 = layer.w13_weight_scale, layer.w2_weight_scale
        a.group13, a.group2 = cfg.hidden_dim // s13.shape[1], I // s2.shape[1]
        tensors = (layer.w13_weight, s13, layer.w2_weight, s2)
        a.w13, a.s13, a.w2, a.s2 = (t.data_ptr() for t in tensors)
        sizes = [(t.numel() * (2 if t.dtype == torch.uint8 else 1), t.dtype) for t in tensors]
    else:
        tensors = (layer.w13_weight, layer.w13_weight_scale_fp32, layer.w2_weight, layer.w2_weight_scale_fp32)
        a.w13, a.s13, a.w2, a.s2 = (t.data_ptr() for t in tensors)
        sizes = [(t.numel(), t.dtype) for t in tensors]
    H = cfg.hidden_dim
    per13, per2 = (H // a.group13, I // a.group2) if a.weights == _INT4 else (1, 1)
    wtype = torch.uint8 if a.weights == _INT4 else torch.int8
    if sizes != [(E * 2 * I * H, wtype), (E * 2 * I * per13, torch.float32), (E * H * I, wtype),
                 (E * H * per2, torch.float32)]:
        return plan  # not laid out (process_weights_after_loading has not run): the operators say what is wrong
    a.pair_order = int(layer.use_pair_order)
    if a.weights == _INT4 or not a.pair_order:
        # the sorting launch's arrival counter, shared with the operator-by-operator path
        counter = getattr(layer, "_small_batch_counter", None)
        if counter is None or counter.device != x.device:
            counter = layer._small_batch_counter = torch.zeros((1,), dtype=torch.int32, device=x.device)
        a.sync_counter = counter.data_ptr()
    if logits is None:
        w, gb = gate.weight, gate.bias
        if tuple(w.shape) != (E, H) or w.dtype != torch.float32 or not w.is_contiguous() or not w.is_cuda:
            return plan
        if gb is not None and (gb.dtype != torch.float32 or gb.numel() != E or not gb.is_contiguous()):
            return plan
        a.gate_weight, a.gate_bias = w.data_ptr(), _ptr(gb)
    if shared is not None:
        h, n = shared.gate_up_weight.shape
        if h != H or n % 2 or tuple(shared.down_weight.shape) != (n // 2, H):
            return plan
        a.shared_intermediate = n // 2
        a.shared = 2 if shared.multistream_overlap else 1
        a.shared_limit, a.shared_alpha, a.shared_beta = (shared.swiglu_limit, shared.swiglu_alpha, shared.swiglu_beta)
        a.shared_w13, a.shared_w2 = shared.gate_up_weight.data_ptr(), shared.down_weight.data_ptr()
        a.shared_s13, a.shared_s2 = shared.gate_up_scale_fp32.data_ptr(), shared.down_scale_fp32.data_ptr()
        if a.shared == 2:
            a.shared_stream = shared_experts_calculation_stream().cuda_stream
    if layer.dynamic_eplb and layer.eplb_heat_collection_status:
        a.load = layer.moe_load.data_ptr()
    plan.desc, plan.ref = a, ctypes.addressof(a)
    plan.hidden, plan.experts = H, E
    plan.forward, plan.workspace = lib.moe355_layer_forward, lib.moe355_layer_workspace
    return plan


def layer_call(layer, x: torch.Tensor, logits: torch.Tensor | None) -> torch.Tensor | None:
    """The layer's output, or None when the call has to go operator by operator (an option the library has no whole
    form for, or arguments that the operators refuse with a message of their own)."""
    key = _key(layer, x.dtype, None if logits is None else logits.dtype)
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
        if logits.shape != (T, plan.experts) or not logits.is_contiguous() or not logits.is_cuda:
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
