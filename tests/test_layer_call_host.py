"""Which calls the whole-layer call takes, and when it looks at the layer again: host code, no GPU."""
import ctypes
import threading
import types

import pytest
import torch

from vllm_ascend_amd import _lib
from vllm_ascend_amd.fused_moe.contracts import FusedMoEConfig
from vllm_ascend_amd.fused_moe.gate_linear import AscendGateLinear
from vllm_ascend_amd.fused_moe.layer import AscendRoutedExperts
from vllm_ascend_amd.fused_moe import layer_call as layer_call_module
from vllm_ascend_amd.fused_moe.layer_call import layer_call
from vllm_ascend_amd.fused_moe.router import AscendFusedTopKRouter
from vllm_ascend_amd.fused_moe.shared_experts import AscendSharedExperts
from vllm_ascend_amd.quantization import get_scheme_class

E, K, H, I = 8, 2, 128, 32


def _layer(scheme="W8A8_DYNAMIC", cls=AscendRoutedExperts, shared=False, gate=False):
    """A layer on the CPU with the attributes that loading its weights leaves behind."""
    layer = cls(FusedMoEConfig(E, K, H, I), get_scheme_class(scheme, "moe")(),
                AscendFusedTopKRouter(K, E, e_score_correction_bias=torch.zeros(E)), params_dtype=torch.float32,
                device="cpu")
    if scheme == "W8A8_DYNAMIC":
        layer.w13_weight_scale_fp32, layer.w2_weight_scale_fp32 = torch.zeros(E, 2 * I), torch.zeros(E, H)
    if shared:
        s = AscendSharedExperts.__new__(AscendSharedExperts)
        torch.nn.Module.__init__(s)
        s.gate_up_weight, s.down_weight = torch.zeros(H, 2 * I, dtype=torch.int8), torch.zeros(I, H, dtype=torch.int8)
        s.gate_up_scale_fp32, s.down_scale_fp32 = torch.zeros(2 * I), torch.zeros(H)
        s.swiglu_limit, s.swiglu_alpha, s.swiglu_beta, s.multistream_overlap = 0.0, 1.0, 0.0, False
        layer.shared_experts = s
    if gate:
        layer.gate = AscendGateLinear(H, E, bias=True, device="cpu")
    return layer


class _Gpu(torch.Tensor):
    """A tensor that says it is on the GPU: nothing here gets as far as a launch."""

    is_cuda = True


X, LOGITS = torch.zeros(3, H, dtype=torch.bfloat16).as_subclass(_Gpu), torch.zeros(3, E).as_subclass(_Gpu)


class _ModuleRouter(torch.nn.Module, AscendFusedTopKRouter):
    def __init__(self):
        torch.nn.Module.__init__(self)
        AscendFusedTopKRouter.__init__(self, K, E)


class _ModuleScheme(torch.nn.Module):
    def __init__(self, scheme):
        super().__init__()
        self.scheme = scheme


def _foreign_parameters(layer):
    p = layer._parameters
    for name in list(p):
        p["expert_" + name] = p.pop(name)


def _set_parameter(layer, name):
    t = torch.nn.Parameter(torch.arange(E), requires_grad=False)
    delattr(layer, name)
    setattr(layer, name, t)


# layers that are put together in other ways than the stock one: none of them is the whole-layer call's, and none of
# them is a reason to raise
FOREIGN = {
    "a shared expert of another class": lambda l: setattr(l, "shared_experts", torch.nn.Linear(2, 2)),
    "a shared expert that is a function": lambda l: setattr(l, "shared_experts", lambda x, quantized=None: x),
    "a router that is a module": lambda l: (delattr(l, "router"), setattr(l, "router", _ModuleRouter())),
    "a scheme that is a module": lambda l: setattr(l, "quant_method", _ModuleScheme(l.__dict__.pop("quant_method"))),
    "other parameter names": _foreign_parameters,
    "log2phy as a parameter": lambda l: _set_parameter(l, "log2phy"),
    "an expert map as a parameter": lambda l: _set_parameter(l, "ascend_expert_map"),
    "weights that have not been laid out": lambda l: delattr(l, "w13_weight_scale_fp32"),
}


@pytest.mark.parametrize("what", list(FOREIGN))
def test_foreign_parts_go_operator_by_operator(what):
    layer = _layer()
    FOREIGN[what](layer)
    assert layer_call(layer, X, LOGITS) is None


def test_a_gate_that_is_any_callable():
    layer = _layer()
    layer.gate = lambda x: (LOGITS, None)
    assert layer_call(layer, X, None) is None
    assert layer_call(layer, X, LOGITS) is None


# ---------------------------------------------------------------- what the library is told
@pytest.fixture
def told(monkeypatch):
    """The descriptions that reach the library, which is not called."""
    calls = []

    def forward(ref, *args):
        calls.append(_lib.Layer.from_buffer_copy(ctypes.string_at(ref, ctypes.sizeof(_lib.Layer))))
        return 0

    lib = types.SimpleNamespace(moe355_layer_forward=forward, moe355_layer_workspace=lambda ref, T: 256)
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(layer_call_module, "_stream", lambda t: 0)
    return calls


def _as_gpu(layer):
    layer.router.e_score_correction_bias = layer.router.e_score_correction_bias.as_subclass(_Gpu)
    if layer.gate is not None:
        for name, p in layer.gate._parameters.items():
            layer.gate._parameters[name] = p.as_subclass(_Gpu)
    return layer


@pytest.fixture(params=["W8A8_DYNAMIC", "W4A8_DYNAMIC"])
def scheme(request):
    return request.param


def _laid_out(scheme="W8A8_DYNAMIC", **kw):
    layer = _layer(scheme, **kw)
    p = layer._parameters
    if scheme == "W8A8_DYNAMIC":
        p["w13_weight"].data, p["w2_weight"].data = (torch.zeros(E, H, 2 * I, dtype=torch.int8),
                                                     torch.zeros(E, I, H, dtype=torch.int8))
    else:
        p["w13_weight"].data, p["w2_weight"].data = (torch.zeros(E, H * I, dtype=torch.uint8),
                                                     torch.zeros(E, H * I // 2, dtype=torch.uint8))
        p["w13_weight_scale"].data, p["w2_weight_scale"].data = torch.zeros(E, 1, 2 * I), torch.zeros(E, 1, H)
    return _as_gpu(layer)


def test_a_laid_out_layer_is_one_call(told, scheme):
    layer = _laid_out(scheme)
    for _ in range(2):
        assert layer_call(layer, X, LOGITS) is not None
    assert len(told) == 2 and told[0].w13 == layer.w13_weight.data_ptr()
    assert told[1].bias == layer.router.e_score_correction_bias.data_ptr()


def test_a_bias_of_another_type_at_the_same_address(told):
    layer = _laid_out()
    layer_call(layer, X, LOGITS)
    fp32 = layer.router.e_score_correction_bias
    half = layer.router.e_score_correction_bias = fp32.view(torch.bfloat16)[:E]
    assert half.data_ptr() == fp32.data_ptr()
    layer_call(layer, X, LOGITS)
    bias = layer.router.e_score_correction_bias
    assert bias.dtype == torch.float32 and told[-1].bias == bias.data_ptr() != half.data_ptr()


def test_a_narrower_gate_weight_at_the_same_address(told):
    layer = _laid_out(gate=True)
    assert layer_call(layer, X, None) is not None
    weight = layer.gate._parameters["weight"]
    layer.gate._parameters["weight"] = weight.view(-1)[: E * H // 2].view(E, H // 2)
    assert layer.gate._parameters["weight"].data_ptr() == weight.data_ptr()
    assert layer_call(layer, X, None) is None  # the gate refuses it


# tensors that the operators convert, copy or refuse: at another address, or at the one that a plan was made with
CHANGED = {
    "weight of another shape": ("w13_weight", lambda t: t.data.view(E, 2 * I, H)),
    "weight that is not contiguous": ("w2_weight", lambda t: torch.zeros(E, H, I, dtype=torch.int8).transpose(1, 2)),
    "scale of another type, same address": ("w13_weight_scale_fp32",
                                            lambda t: t.view(torch.float16)[:, : 2 * I].reshape(-1)[: E * 2 * I]),
    "scale of another type": ("w2_weight_scale_fp32", lambda t: t.double()),
    "scale with too few values": ("w2_weight_scale_fp32", lambda t: t[: E // 2]),
    "scale that is not contiguous": ("w2_weight_scale_fp32", lambda t: torch.zeros(H, E).t()),
}


@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("what", list(CHANGED))
def test_tensors_the_library_cannot_read(told, what, planned):
    layer = _laid_out()
    if planned:
        assert layer_call(layer, X, LOGITS) is not None
    name, change = CHANGED[what]
    if name in layer._parameters:
        layer._parameters[name].data = change(layer._parameters[name])
    else:
        setattr(layer, name, change(getattr(layer, name)))
    assert layer_call(layer, X, LOGITS) is None


SHARED_CHANGED = {
    "weight that is not contiguous": ("gate_up_weight", lambda t: torch.zeros(2 * I, H, dtype=torch.int8).t()),
    "weight of another type": ("down_weight", lambda t: t.to(torch.int32)),
    "scale of another type": ("down_scale_fp32", lambda t: t.half()),
    "scale with too few values": ("gate_up_scale_fp32", lambda t: t[:I]),
}


@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("what", list(SHARED_CHANGED))
def test_shared_expert_tensors_the_library_cannot_read(told, what, planned):
    layer = _laid_out(shared=True)
    if planned:
        assert layer_call(layer, X, LOGITS) is not None
    name, change = SHARED_CHANGED[what]
    setattr(layer.shared_experts, name, change(getattr(layer.shared_experts, name)))
    assert layer_call(layer, X, LOGITS) is None


# ---------------------------------------------------------------- methods of the caller's in the layer
def _wrapped(obj, name):
    fn = getattr(obj, name)
    setattr(obj, name, lambda *a, **kw: fn(*a, **kw))


REPLACED = {
    "router.select_experts": lambda l: _wrapped(l.router, "select_experts"),
    "router.is_fused_supported": lambda l: _wrapped(l.router, "is_fused_supported"),
    "quant_method.apply_small_batch": lambda l: _wrapped(l.quant_method, "apply_small_batch"),
    "moe_comm_method.finalize": lambda l: _wrapped(l.moe_comm_method, "finalize"),
    "prepare_finalize.prepare": lambda l: _wrapped(l.moe_comm_method.prepare_finalize, "prepare"),
    "shared_experts.forward": lambda l: _wrapped(l.shared_experts, "forward"),
    "a hook of the shared expert": lambda l: l.shared_experts.register_forward_hook(lambda *a: None),
    "gate.forward": lambda l: _wrapped(l.gate, "forward"),
    "a hook of the gate": lambda l: l.gate.register_forward_pre_hook(lambda *a: None),
}


@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("what", list(REPLACED))
def test_replaced_methods_are_not_passed_by(told, what, planned):
    layer = _laid_out(shared=True, gate=True)
    if planned:
        assert layer_call(layer, X, None) is not None
    REPLACED[what](layer)
    assert layer_call(layer, X, None) is None


@pytest.mark.parametrize("cls, name", [(AscendFusedTopKRouter, "select_experts"), (AscendSharedExperts, "forward"),
                                       (AscendGateLinear, "forward"),
                                       (get_scheme_class("W8A8_DYNAMIC", "moe"), "apply_small_batch")])
def test_patched_classes_are_not_passed_by(told, monkeypatch, cls, name):
    layer = _laid_out(shared=True, gate=True)
    assert layer_call(layer, X, None) is not None
    fn = getattr(cls, name)
    monkeypatch.setattr(cls, name, lambda *a, **kw: fn(*a, **kw))
    assert layer_call(layer, X, None) is None


@pytest.mark.parametrize("name", ["forward_impl", "_run_experts", "_record_expert_load"])
@pytest.mark.parametrize("where", ["subclass", "instance", "class"])
def test_a_layer_with_a_form_of_its_own(told, monkeypatch, name, where):
    class Own(AscendRoutedExperts):
        pass

    layer = _laid_out(cls=Own)
    assert layer(X, LOGITS) is not None and len(told) == 1  # a subclass alone changes nothing
    owner = {"subclass": Own, "instance": layer, "class": AscendRoutedExperts}[where]
    seen = []
    result = types.SimpleNamespace(routed_out=X)
    monkeypatch.setattr(owner, name, lambda *a, **kw: seen.append(name) or result)
    if name == "_record_expert_load":  # called behind the operators, which the library of this test does not have
        with pytest.raises(AttributeError, match="moe355_"):
            layer(X, LOGITS)
    else:
        assert layer(X, LOGITS) is X and seen == [name]
    assert len(told) == 1


def test_routers_that_select_by_themselves():
    from vllm_ascend_amd.fused_moe.router import replaces_selection

    class Sub(AscendFusedTopKRouter):
        pass

    class Own(AscendFusedTopKRouter):
        def _compute_routing(self, *a, **kw):
            return super()._compute_routing(*a, **kw)

    assert not replaces_selection(AscendFusedTopKRouter(K, E)) and not replaces_selection(Sub(K, E))
    assert not replaces_selection(types.SimpleNamespace(top_k=K))  # numbers alone
    assert replaces_selection(Own(K, E)) and replaces_selection(types.SimpleNamespace(select_experts=None))
    router = AscendFusedTopKRouter(K, E)
    _wrapped(router, "select_experts")
    assert replaces_selection(router)


# ---------------------------------------------------------------- state that calls would share
@pytest.mark.parametrize("pair_order", [True, False])
def test_no_counter_is_shared_between_calls(told, scheme, pair_order):
    """A launch that counts its workgroups on device memory must not share it with one that may run at the same time:
    the layer has no such memory, whatever form it takes."""
    layer = _laid_out(scheme)
    layer.use_pair_order = pair_order
    assert layer_call(layer, X, LOGITS) is not None
    assert not told[-1].sync_counter


def test_each_thread_waits_for_its_own_shared_expert(monkeypatch):
    """Two calls of one layer at a time, the shared expert of both on the side stream: neither takes the other's event."""
    here = threading.local()

    class Stream:
        def __init__(self, name):
            self.name, self.waited = name, []

        def record_event(self):
            return f"{here.name} on {self.name}"

        def wait_event(self, evt):
            self.waited.append(evt)

        def __enter__(self):
            return self

        def __exit__(self, *exc):
            return None

    side = Stream("side")
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: here.stream)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: s)
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda self, s: None)
    monkeypatch.setattr("vllm_ascend_amd.fused_moe.shared_experts.shared_experts_calculation_stream",
                        lambda *a: side)
    monkeypatch.setattr(AscendSharedExperts, "_mlp", lambda self, x, quantized=None: x)
    shared = AscendSharedExperts.__new__(AscendSharedExperts)
    torch.nn.Module.__init__(shared)
    shared.multistream_overlap, shared._done_evts = True, {}
    both_enqueued, waited = threading.Barrier(2, timeout=30), {}

    def call(name):
        here.name, here.stream = name, Stream(name)
        shared.forward(torch.zeros(1))
        both_enqueued.wait()
        shared.wait()
        shared.wait()  # nothing left
        waited[name] = here.stream.waited

    threads = [threading.Thread(target=call, args=(n,)) for n in ("a", "b")]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert waited == {"a": ["a on side"], "b": ["b on side"]}


def test_every_device_has_a_side_stream_of_its_own(monkeypatch):
    from vllm_ascend_amd.fused_moe import shared_experts as module

    monkeypatch.setattr(module, "_SIDE_STREAMS", {})
    monkeypatch.setattr(torch.cuda, "Stream", lambda device=None: types.SimpleNamespace(device=device))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    first, second = module.shared_experts_calculation_stream(0), module.shared_experts_calculation_stream(1)
    assert (first.device, second.device) == (0, 1)
    assert module.shared_experts_calculation_stream() is second and module.shared_experts_calculation_stream(0) is first
