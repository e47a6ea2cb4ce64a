"""The layer as one native call (``moe355_layer_forward``): the same operators, chosen by the same rules, as
``AscendRoutedExperts.forward_impl`` (``vllm_ascend/ops/fused_moe/routed_experts.py:496-609``) enqueues one by one, so
the output is the same, bit for bit.

A decode step of a small layer is bound by the host: going operator by operator costs 50 to 240 us of interpreter,
allocations and event records for 27 to 200 us of kernels.  Here a call is two allocations and one foreign call; what
the library needs to know about the layer is gathered once and kept until something about the layer changes."""
from __future__ import annotations

import ctypes

import torch

from .. import _lib
from ..kernels import _DT, _stream
from .gate_linear import AscendGateLinear
from .moe_comm_method import AllGatherCommImpl, _IdentityPrepareFinalize
from .router import AscendFusedTopKRouter
from .shared_experts import AscendSharedExperts, shared_experts_calculation_stream

_MAX_SIZES = 256  # batch sizes whose scratch size is remembered


class _Plan:
    """What one layer looks like to the library; ``desc`` is None when the native call cannot take it."""

    __slots__ = ("key", "desc", "ref", "hidden", "experts", "sizes", "keep", "forward", "workspace")

    def __init__(self, key):
        self.key = key
        self.desc = self.ref = None
        self.sizes = {}

    def __reduce__(self):  # a copied or pickled layer makes its own
        return type(None), ()


def _ptr(t):
    return None if t is None else t.data_ptr()


def _key(layer, d, x_dtype, logits_dtype):
    """Everything the plan was made from.  Compared on every call, so plain dictionary lookups."""
    p, b, m = d["_parameters"], d["_buffers"], d["_modules"]
    q, r, gate, shared = d["quant_method"], d["router"], m.get("gate", d.get("gate")), m.get("shared_experts", d.get("shared_experts"))
    qd, rd = q.__dict__, r.__dict__
    bias = rd.get("e_score_correction_bias")
    if qd.get("use_expert_weight_list") and "w13_weight_list" in d:
        w = tuple(d[n].table.data_ptr() for n in ("w13_weight_list", "w13_weight_scale_fp32_list", "w2_weight_list",
                                                  "w2_weight_scale_list"))
    else:
        w = [p["w13_weight"].data_ptr(), p["w2_weight"].data_ptr()]
        for n in ("w13_weight_scale_fp32", "w2_weight_scale_fp32"):
            t = d.get(n)
            w.append(0 if t is None else t.data_ptr())
        for n in ("w13_weight_scale", "w2_weight_scale"):
            w.append(p[n].data_ptr())
    sh = g = None
    if shared is not None:
        s = shared.__dict__
        sh = (id(shared), type(shared), s["multistream_overlap"], s["swiglu_limit"], s["swiglu_alpha"],
              s["swiglu_beta"], s["gate_up_weight"].data_ptr(), s["down_weight"].data_ptr(),
              s["gate_up_scale_fp32"].data_ptr(), s["down_scale_fp32"].data_ptr(),
              bool(s["_forward_hooks"] or s["_forward_pre_hooks"]))
    if gate is not None:
        s = gate.__dict__
        gp = s["_parameters"]
        g = (id(gate), type(gate), _ptr(gp.get("weight")), _ptr(gp.get("bias")),
             bool(s["_forward_hooks"] or s["_forward_pre_hooks"]))
    load = b.get("moe_load")
    return (x_dtype, logits_dtype, w, sh, g, q, type(q), qd.get("in_dtype"), qd.get("group_size"), r, type(r),
            rd.get("top_k"), rd.get("renormalize"), rd.get("num_expert_group"), rd.get("topk_group"),
            rd.get("scoring_func"), rd.get("routed_scaling_factor"), 0 if bias is None else bias.data_ptr(),
            d["activation"], d["apply_router_weight_on_input"], d["ascend_expert_map"] is None,
            d["global_redundant_expert_num"], d["ascend_mc2_mask"] is None, d["ascend_pertoken_scale"] is None,
            d["enable_force_load_balance"], d["log2phy"] is None and b.get("log2phy") is None,
            d["use_fused_small_batch"], d["use_pair_order"], d["dynamic_eplb"], d["eplb_heat_collection_status"],
            0 if load is None else load.data_ptr(), d["moe_config"], d["moe_config"].swiglu_limit,
            d["moe_comm_method"])


def _supported(layer, gate, shared, x, logits) -> bool:
    """The calls ``supports_small_batch`` takes (per-expert weight lists too), with the stock parts around them."""
    from ..quantization.w4a8 import AscendW4A8DynamicFusedMoEMethod
    from ..quantization.w8a8_dynamic import AscendW8A8DynamicFusedMoEMethod

    q, r, comm = layer.quant_method, layer.router, layer.moe_comm_method
    if getattr(q, "use_expert_weight_list", False) and not hasattr(layer, "w13_weight_list"):
        return False
    if type(q) not in (AscendW8A8DynamicFusedMoEMethod, AscendW4A8DynamicFusedMoEMethod):
        return False
    if type(q) is AscendW4A8DynamicFusedMoEMethod and q.use_expert_weight_list:
        return False
    if type(r) is not AscendFusedTopKRouter or not r.is_fused_supported(x):
        return False
    if type(comm) is not AllGatherCommImpl or type(comm.prepare_finalize) is not _IdentityPrepareFinalize:
        return False
    if x.dtype not in (torch.bfloat16, torch.float16) or x.dtype != q.in_dtype or not layer.use_fused_small_batch:
        return False
    if (layer.apply_router_weight_on_input or layer.ascend_pertoken_scale is not None
            or layer.ascend_expert_map is not None or layer.ascend_mc2_mask is not None
            or layer.global_redundant_expert_num or layer.enable_force_load_balance or layer.log2phy is not None):
        return False
    act = layer.activation
    if (getattr(act, "value", act) or "silu") != "silu":
        return False
    if logits is not None and logits.dtype not in _DT:
        return False
    if logits is None and (type(gate) is not AscendGateLinear or gate._forward_hooks or gate._forward_pre_hooks):
        return False
    if shared is not None and (type(shared) is not AscendSharedExperts or shared._forward_hooks
                               or shared._forward_pre_hooks):
        return False
    if layer.dynamic_eplb and layer.eplb_heat_collection_status and layer.multi_stage:
        return False  # one row of loads per pass, indexed on the device: operator by operator
    E, bias = layer.moe_config.num_experts, r.e_score_correction_bias
    return bias is None or (bias.dim() == 1 and bias.numel() == E and bias.is_contiguous() and bias.is_cuda)


def _make_plan(layer, d, x, logits) -> _Plan:
    m = d["_modules"]
    gate = m.get("gate", d.get("gate"))
    shared = m.get("shared_experts", d.get("shared_experts"))
    logits_dtype = torch.float32 if logits is None else logits.dtype
    r = layer.router
    supported = _supported(layer, gate, shared, x, logits)
    bias = r.e_score_correction_bias if supported else None
    if bias is not None and bias.dtype != logits_dtype:
        bias = r.e_score_correction_bias = bias.to(logits_dtype)
    plan = _Plan(_key(layer, d, x.dtype, None if logits is None else logits.dtype))
    if not supported:
        return plan
    q, cfg, lib = layer.quant_method, layer.moe_config, _lib.load()
    E, I = cfg.num_experts, cfg.intermediate_size_per_partition
    a = _lib.Layer()
    a.hidden, a.intermediate, a.num_experts, a.top_k = cfg.hidden_dim, I, E, r.top_k
    a.k_group = r.topk_group if r.topk_group is not None else 1
    a.group_count = r.num_expert_group if r.num_expert_group is not None else 1
    a.renorm, a.norm_type = int(r.renormalize), 0 if r.scoring_func == "softmax" else 1
    a.routed_scaling_factor, a.eps, a.swiglu_limit = r.routed_scaling_factor, 1e-20, cfg.swiglu_limit or 0.0
    a.x_dtype, a.bias = _DT[x.dtype], _ptr(bias)
    if q.use_expert_weight_list:
        lists = (layer.w13_weight_list, layer.w13_weight_scale_fp32_list, layer.w2_weight_list,
                 layer.w2_weight_scale_list)
        a.weights = 1
        a.w13, a.s13, a.w2, a.s2 = (t.table.data_ptr() for t in lists)
        sizes = [(t[0].numel() * len(t), t[0].dtype) for t in lists]
    elif hasattr(q, "group_size"):
        s13, s2 = layer.w13_weight_scale, layer.w2_weight_scale
        a.weights, a.group13, a.group2 = 2, cfg.hidden_dim // s13.shape[1], I // s2.shape[1]
        tensors = (layer.w13_weight, s13, layer.w2_weight, s2)
        a.w13, a.s13, a.w2, a.s2 = (t.data_ptr() for t in tensors)
        sizes = [(t.numel() * (2 if t.dtype == torch.uint8 else 1), t.dtype) for t in tensors]
    else:
        tensors = (layer.w13_weight, layer.w13_weight_scale_fp32, layer.w2_weight, layer.w2_weight_scale_fp32)
        a.w13, a.s13, a.w2, a.s2 = (t.data_ptr() for t in tensors)
        sizes = [(t.numel(), t.dtype) for t in tensors]
    H = cfg.hidden_dim
    per13, per2 = (H // a.group13, I // a.group2) if a.weights == 2 else (1, 1)
    wtype = torch.uint8 if a.weights == 2 else torch.int8
    if sizes != [(E * 2 * I * H, wtype), (E * 2 * I * per13, torch.float32), (E * H * I, wtype),
                 (E * H * per2, torch.float32)]:
        return plan  # not laid out (process_weights_after_loading has not run): the operators say what is wrong
    a.pair_order = int(layer.use_pair_order)
    if a.weights == 2 or not a.pair_order:
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
    d = layer.__dict__
    plan = d.get("_layer_plan")
    if plan is None or plan.key != _key(layer, d, x.dtype, None if logits is None else logits.dtype):
        if not x.is_cuda or x.dim() != 2:
            return None
        plan = d["_layer_plan"] = _make_plan(layer, d, x, logits)
    if plan.desc is None:
        return None
    shape = x.shape
    if len(shape) != 2 or shape[1] != plan.hidden or not x.is_cuda or not x.is_contiguous():
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
