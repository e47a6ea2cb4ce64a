"""Which calls the whole-layer call takes, and when it looks at the layer again: host code, no GPU."""
import torch

import pytest

from vllm_ascend_amd.fused_moe.contracts import FusedMoEConfig
from vllm_ascend_amd.fused_moe.gate_linear import AscendGateLinear
from vllm_ascend_amd.fused_moe.layer import AscendRoutedExperts
from vllm_ascend_amd.fused_moe.layer_call import layer_call
from vllm_ascend_amd.fused_moe.router import AscendFusedTopKRouter
from vllm_ascend_amd.fused_moe.shared_experts import AscendSharedExperts
from vllm_ascend_amd.quantization import get_scheme_class

E, K, H, I = 8, 2, 64, 32


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
