"""CPU-side checks: the C-ABI library loads and exports every symbol the header declares, the host
mirror of the reference interface behaves like the reference for argument handling, and nothing in
the package reaches into the checker."""
import ctypes
import json
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KATS = json.load(open(os.path.join(ROOT, "tests", "golden", "reference_kats.json")))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "moe355.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(moe355_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from vllm_ascend_amd import _lib

    lib = ctypes.CDLL(_lib.LIB_PATH)
    names = _declared_symbols()
    assert len(names) >= 15
    for name in names:
        assert hasattr(lib, name), f"{name} is declared in include/moe355.h but not exported"
    # the ctypes prototypes cover the same set
    assert sorted(_lib.PROTOTYPES) == names


def test_abi_version_and_strerror():
    from vllm_ascend_amd import _lib

    lib = _lib.load()
    assert lib.moe355_abi_version() == _lib.ABI_VERSION
    assert lib.moe355_strerror(0) == b"ok"
    assert b"workspace" in lib.moe355_strerror(-3)


def test_argument_validation_without_gpu():
    """Rejections happen on the host before any launch, so they can be exercised without a GPU."""
    from vllm_ascend_amd import _lib

    lib = _lib.load()
    one = ctypes.c_void_p(256)  # never dereferenced: every call below is refused first
    assert lib.moe355_dynamic_quant(one, 1, -1, 8, one, one, None) == -1
    assert lib.moe355_dynamic_quant(one, 0, 4, 8, one, one, None) == -5  # fp32 input not supported
    assert lib.moe355_gating_top_k(one, 0, None, 4, 4096, 8, 1, 1, 1, 1, 0, 0, 1.0, 1e-20, one, one, None, None, 0,
                                   None) == -2  # E > 2048
    assert lib.moe355_gating_top_k(one, 0, None, 4, 64, 8, 1, 3, 1, 1, 0, 0, 1.0, 1e-20, one, one, None, None, 0,
                                   None) == -2  # E % group_count
    assert lib.moe355_gating_top_k(one, 0, None, 4, 64, 8, 1, 1, 1, 1, 2, 0, 1.0, 1e-20, one, one, None, None, 0,
                                   None) == -1  # norm_type
    assert lib.moe355_gmm_i32(one, one, one, 0, 4, 48, 64, 2, one, one, 256, None) == -2  # K % 32
    assert lib.moe355_gmm_i32(one, one, one, 7, 4, 64, 64, 2, one, one, 256, None) == -1  # group list type
    assert lib.moe355_gmm1_swiglu_quant(one, one, one, one, one, 0, 4, 64, 64, 2, 0.0, one, one, None, 0,
                                        None) == -3  # no workspace
    assert lib.moe355_init_routing(one, 1, 4, 64, one, 2, 8, 5, 1, one, one, one, one, one, 1 << 20, None) == -5
    assert lib.moe355_format_cast_nz(one, 0, 2, 48, 64, one, None) == -2
    assert lib.moe355_token_unpermute(one, 0, one, one, 4, 2, 64, 8, None, one, None) == -5
    assert lib.moe355_init_routing_workspace(64, 8, 128) >= 128 * 4 + 129 * 4
    assert lib.moe355_gmm1_swiglu_quant_workspace(512, 1536, 2048, 128) >= 512 * 768 * 4


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    from vllm_ascend_amd import _lib

    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libmoe355.so"))
    with pytest.raises(ImportError, match="no CPU or PyTorch fallback"):
        _lib.load()


def test_package_never_touches_the_checker():
    pkg = os.path.join(ROOT, "vllm_ascend_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                text = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in text.lower(), f"{f} mentions the checker"


def test_custom_ops_schemas_and_meta():
    from vllm_ascend_amd.custom_ops import enable_custom_op

    assert enable_custom_op()
    ops = torch.ops._C_ascend
    x = torch.empty(5, 128, device="meta")
    y, idx, out = ops.moe_gating_top_k(x, k=8, k_group=1, group_count=1, group_select_mode=1, renorm=1, norm_type=0,
                                       out_flag=False, routed_scaling_factor=1.0, eps=1e-20, bias_opt=None)
    assert y.shape == (5, 8) and idx.dtype == torch.int32 and out.shape == (5, 128) and out.dtype == torch.float32
    xi = torch.empty(16, 64, dtype=torch.int8, device="meta")
    w = torch.empty(4, 64, 128, dtype=torch.int8, device="meta")
    o, s, off = ops.grouped_matmul_swiglu_quant_weight_nz(
        x=xi, weight=w, weight_scale=torch.empty(4, 128, device="meta"), x_scale=torch.empty(16, device="meta"),
        group_list=torch.empty(4, dtype=torch.int64, device="meta"))
    assert o.shape == (16, 64) and o.dtype == torch.int8 and s.shape == (16,) and s.dtype == torch.float32
    o, s = ops.npu_dequant_swiglu_quant(torch.empty(3, 256, dtype=torch.int32, device="meta"), quant_mode=1)
    assert o.shape == (3, 128) and s.shape == (3,)
    # CPU tensors are refused: only the HIP kernels exist
    with pytest.raises(NotImplementedError):
        ops.moe_gating_top_k(torch.zeros(5, 128), k=8, k_group=1, group_count=1, group_select_mode=1, renorm=1,
                             norm_type=0, out_flag=False, routed_scaling_factor=1.0, eps=1e-20)


def test_gating_argument_checks_match_the_reference_adapter():
    """Messages of csrc/moe/moe_gating_top_k/moe_gating_top_k_torch_adpt.h:33-48."""
    from vllm_ascend_amd.custom_ops import _check_gating

    with pytest.raises(RuntimeError, match="The x should be 2D"):
        _check_gating(torch.zeros(8), None)
    with pytest.raises(RuntimeError, match="tensor expected but got a tensor with dtype"):
        _check_gating(torch.zeros(2, 8, dtype=torch.int32), None)
    with pytest.raises(RuntimeError, match="The dtype of x and bias should be same"):
        _check_gating(torch.zeros(2, 8), torch.zeros(8, dtype=torch.bfloat16))
    with pytest.raises(RuntimeError, match="The bias should be 1D"):
        _check_gating(torch.zeros(2, 8), torch.zeros(1, 8))
    with pytest.raises(RuntimeError, match="The bias first dim should be same as x second dim"):
        _check_gating(torch.zeros(2, 8), torch.zeros(4))


def test_cumsum_group_list_known_answers():
    """Vectors of tests/ut/ops/test_moe_mlp.py:31-62."""
    from vllm_ascend_amd.fused_moe.moe_mlp import cumsum_group_list

    k = KATS["cumsum_group_list"]
    lists = {0: torch.tensor(k["type0_cumsum"]), 1: torch.tensor(k["type1_count"]),
             2: torch.tensor([[1, 2], [2, 1], [0, 0], [0, 0]])}
    for src, dst in k["supported"]:
        assert torch.equal(cumsum_group_list(lists[src], src, dst, expert_num=4), lists[dst])
    with pytest.raises(ValueError, match=r"group_list_type should be in \[0, 1, 2\], but received"):
        cumsum_group_list(lists[0], 4, 0)
    for src, dst in k["unsupported"]:
        with pytest.raises(NotImplementedError, match="This feature is under development."):
            cumsum_group_list(lists[0], src, dst)
    # sparse pairs -> running sum
    sparse = torch.tensor([[1, 2], [3, 1]])
    assert cumsum_group_list(sparse, 2, 0, active_num=3, expert_num=4).tolist() == [0, 2, 2, 3]


def test_scheme_weight_specs_match_the_reference():
    """Names and shapes of vllm_ascend/quantization/methods/w8a8_dynamic.py:198-222."""
    from vllm_ascend_amd.quant_type import QuantType
    from vllm_ascend_amd.quantization import get_scheme_class

    scheme = get_scheme_class("W8A8_DYNAMIC", "moe")()
    assert scheme.quant_type == QuantType.W8A8 and scheme.supports_eplb
    w = scheme.get_weight(8, 1408, 1024, torch.bfloat16)
    assert w["w13_weight"].shape == (8, 2816, 1024) and w["w13_weight"].dtype == torch.int8
    assert w["w2_weight"].shape == (8, 1024, 1408) and w["w2_weight"].dtype == torch.int8
    q = scheme.get_dynamic_quant_param(8, 1408, 1024, torch.bfloat16)
    assert q["w13_weight_scale"].shape == (8, 2816, 1) and q["w13_weight_scale"].dtype == torch.bfloat16
    assert q["w2_weight_scale"].shape == (8, 1024, 1) and q["w13_weight_offset"].shape == (8, 2816, 1)
    with pytest.raises(NotImplementedError):
        get_scheme_class("W8A8_MXFP8", "moe")


def test_unsupported_options_raise_by_name():
    from vllm_ascend_amd.fused_moe.contracts import FusedMoEConfig, build_fused_experts_input, build_token_dispatch_input
    from vllm_ascend_amd.fused_moe.token_dispatcher import TokenDispatcherWithAllGather
    from vllm_ascend_amd.quant_type import QuantType

    with pytest.raises(NotImplementedError, match="one GPU"):
        FusedMoEConfig(num_experts=8, experts_per_token=2, hidden_dim=64, intermediate_size_per_partition=64,
                       ep_size=2)
    disp = TokenDispatcherWithAllGather(top_k=2, num_experts=8, num_local_experts=8)
    base = dict(hidden_states=torch.zeros(4, 64, dtype=torch.bfloat16), topk_weights=torch.zeros(4, 2),
                topk_ids=torch.zeros(4, 2, dtype=torch.int32), w1=[None], w2=[None], quant_type=QuantType.W8A8)
    for kw, pat in ((dict(expert_map=torch.arange(8)), "expert_map"), (dict(mc2_mask=torch.ones(4)), "mc2_mask")):
        inp = build_token_dispatch_input(fused_experts_input=build_fused_experts_input(**base, **kw))
        with pytest.raises(NotImplementedError, match=pat):
            disp.token_dispatch(inp)
    # pertoken_scale is honoured, for the int8 hidden states it belongs to (moe_mlp.py:226-242)
    inp = build_token_dispatch_input(fused_experts_input=build_fused_experts_input(
        **base, pertoken_scale=torch.ones(4)))
    with pytest.raises(ValueError, match="int8 hidden states"):
        disp.token_dispatch(inp)
    from vllm_ascend_amd.fused_moe.moe_mlp import quant_apply_mlp

    with pytest.raises(NotImplementedError, match="relu2"):
        quant_apply_mlp(torch.zeros(1, 8), None, None, None, None, torch.zeros(1), activation="relu2")
    with pytest.raises(NotImplementedError, match="swigluoai"):
        quant_apply_mlp(torch.zeros(1, 8), None, None, None, None, torch.zeros(1), activation="gelu", swiglu_alpha=1.7)


def test_bench_refuses_more_than_one_gpu():
    import subprocess
    import sys

    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode != 0 and "ONE GPU" in r.stderr


def test_w4a8_scheme_specs_and_argument_checks():
    """Parameter names of vllm_ascend/quantization/methods/w4a8.py:146-196 (one int4 value per int8) with the
    group dimension of the scales last; group sizes the kernels cannot take are refused at construction."""
    from vllm_ascend_amd.quant_type import QuantType
    from vllm_ascend_amd.quantization import get_scheme_class

    cls = get_scheme_class("W4A8_DYNAMIC", "moe")
    scheme = cls(group_size=256)
    assert scheme.quant_type == QuantType.W4A8
    w = scheme.get_weight(4, 512, 1024, torch.bfloat16)
    assert w["w13_weight"].shape == (4, 1024, 1024) and w["w13_weight"].dtype == torch.int8
    assert w["w2_weight"].shape == (4, 1024, 512)
    q = scheme.get_dynamic_quant_param(4, 512, 1024, torch.bfloat16)
    assert q["w13_weight_scale"].shape == (4, 1024, 4) and q["w2_weight_scale"].shape == (4, 1024, 2)
    q0 = cls(group_size=0).get_dynamic_quant_param(4, 512, 1024, torch.bfloat16)
    assert q0["w13_weight_scale"].shape == (4, 1024, 1) and q0["w2_weight_scale"].shape == (4, 1024, 1)
    for bad in (-64, 32, 100):
        with pytest.raises(ValueError, match="group_size"):
            cls(group_size=bad)


def test_dense_quant_matmul_argument_checks():
    """npu_quant_matmul stands in for the call in vllm_ascend/ops/fused_moe/shared_experts.py:262-301: what it
    cannot do is refused by name before any kernel is launched."""
    from vllm_ascend_amd import npu_ops

    x = torch.zeros(2, 64, dtype=torch.int8)
    w = torch.zeros(64, 128, dtype=torch.int8)
    s = torch.ones(128)
    with pytest.raises(NotImplementedError, match="offset / bias"):
        npu_ops.npu_quant_matmul(x, w, s, bias=torch.zeros(128))
    with pytest.raises(NotImplementedError, match="int8"):
        npu_ops.npu_quant_matmul(x.to(torch.bfloat16), w, s)
    with pytest.raises(NotImplementedError, match="pertoken_scale"):
        npu_ops.npu_quant_matmul(x, w, s, output_dtype=torch.bfloat16)
    with pytest.raises(NotImplementedError, match="output_dtype"):
        npu_ops.npu_quant_matmul(x, w, s, pertoken_scale=torch.ones(2), output_dtype=torch.float32)
    with pytest.raises(RuntimeError):   # CPU tensors never reach a kernel: there is no host fallback
        npu_ops.npu_quant_matmul(x, w, s, output_dtype=torch.int32)


def test_grouped_gemm_launchers_check_their_operands_on_the_host():
    """The C ABI takes raw pointers: a scale in the model dtype, a short group list or a mis-shaped x must raise
    in Python instead of being read out of bounds on the device.  (The checks run before the device test, so
    CPU tensors reach them.)"""
    from vllm_ascend_amd import kernels as K

    E, n, k, rows = 4, 128, 64, 8
    x = torch.zeros(rows, k, dtype=torch.int8)
    w = torch.zeros(E, k, n, dtype=torch.int8)
    s = torch.ones(E, n)
    xs = torch.ones(rows)
    gl = torch.tensor([2, 2, 2, 2])
    good = dict(x=x, weight_nz=w, weight_scale=s, x_scale=xs, group_list=gl)

    def gmm1(**kw):
        a = {**good, **kw}
        return K.gmm1_swiglu_quant(a["x"], a["weight_nz"], a["weight_scale"], a["x_scale"], a["group_list"], 1, n, k)

    with pytest.raises(TypeError, match="x must be int8"):
        gmm1(x=x.to(torch.bfloat16))
    with pytest.raises(ValueError, match=r"x must be \[rows, K"):
        gmm1(x=torch.zeros(rows, k + 32, dtype=torch.int8))
    with pytest.raises(ValueError, match="one entry per expert"):
        gmm1(group_list=gl[:3])
    with pytest.raises(TypeError, match="x_scale must be float32"):
        gmm1(x_scale=xs.to(torch.bfloat16))
    with pytest.raises(ValueError, match="one scale per row"):
        gmm1(x_scale=torch.ones(rows - 1))
    with pytest.raises(TypeError, match="weight scale must be float32"):
        gmm1(weight_scale=s.to(torch.bfloat16))
    with pytest.raises(ValueError, match="weight scale holds"):
        gmm1(weight_scale=torch.ones(E, n // 2))
    with pytest.raises(ValueError, match="weight holds"):
        gmm1(weight_nz=torch.zeros(E, k, n // 2, dtype=torch.int8))
    with pytest.raises(RuntimeError, match="no CPU implementation"):  # everything else right: refused as a CPU tensor
        gmm1()
    w2 = torch.zeros(E, n // 2, 64, dtype=torch.int8)
    q1 = torch.zeros(rows, n // 2, dtype=torch.int8)
    with pytest.raises(TypeError, match="per_token_scale must be float32"):
        K.gmm2_dequant(q1, w2, torch.ones(E, 64), xs.double(), gl, 1, 64, n // 2)
    with pytest.raises(ValueError, match="one entry per expert"):
        K.gmm2_dequant(q1, w2, torch.ones(E, 64), xs, gl[:2], 1, 64, n // 2)
    with pytest.raises(TypeError, match="weight scale must be float32"):
        K.gmm2_dequant(q1, w2, torch.ones(E, 64, dtype=torch.bfloat16), xs, gl, 1, 64, n // 2)
    w4 = torch.zeros(E, n * k // 2, dtype=torch.uint8)
    with pytest.raises(ValueError, match="weight scale holds"):
        K.gmm1_swiglu_quant_w4(x, w4, torch.ones(E, 1, n), 32, xs, gl, 1, n, k)  # group 32: two groups expected


def test_expert_tensor_lists_keep_their_address_tables():
    """One table per list, built when the list is created and kept for its lifetime (a captured HIP graph holds the
    table's address): many layers, and many lookups, never rebuild or evict a table; replacing an expert rewrites
    one entry of the same table."""
    from vllm_ascend_amd.kernels import ExpertTensorList, _as_expert_list

    layers = []
    for layer in range(40):  # more per-expert-list layers than Qwen3-30B-A3B or DeepSeek-V3 ever evicted before
        lists = [ExpertTensorList([torch.zeros(8, 16, dtype=torch.int8) for _ in range(6)], "w") for _ in range(4)]
        layers.append((lists, [lst.table for lst in lists]))
    for _ in range(3):
        for lists, tables in layers:
            for lst, tab in zip(lists, tables):
                assert _as_expert_list(lst, "w", torch.int8) is lst and lst.table is tab
                assert tab.tolist() == [t.data_ptr() for t in lst]
    lst, tab = layers[0][0][0], layers[0][1][0]
    new = torch.ones(8, 16, dtype=torch.int8)
    lst[2] = new
    assert lst.table is tab and tab[2].item() == new.data_ptr() and lst[2] is new
    with pytest.raises(RuntimeError, match=r"one\s+shape"):
        lst[1] = torch.ones(8, 8, dtype=torch.int8)
    with pytest.raises(TypeError, match="fixed"):
        lst.append(new)
    # a plain list gets a table of its own, for the one call
    plain = [torch.zeros(8, 16, dtype=torch.int8) for _ in range(3)]
    assert isinstance(_as_expert_list(plain, "w", torch.int8), ExpertTensorList)
    with pytest.raises(RuntimeError, match="must be torch.float32"):
        _as_expert_list(lst, "w", torch.float32)


def test_force_load_balance_replaces_the_ids_only():
    """Profile-run routing (vllm_ascend/ops/fused_moe/routed_experts.py:484-492): k distinct random experts per
    token; exercised here on the replacement step itself (the gating kernel needs the GPU)."""
    from vllm_ascend_amd.fused_moe.router import AscendFusedTopKRouter

    r = AscendFusedTopKRouter(4, 32)
    w = torch.rand(10, 4).to(torch.bfloat16)
    ids = torch.zeros(10, 4, dtype=torch.int32)
    r._compute_routing = lambda *a, **k: (w, ids)
    torch.manual_seed(0)
    w2, ids2 = r.select_experts(torch.zeros(10, 8, dtype=torch.bfloat16), torch.zeros(10, 32),
                                enable_force_load_balance=True)
    assert torch.equal(w2, w) and ids2.dtype == ids.dtype and ids2.shape == ids.shape
    assert int(ids2.min()) >= 0 and int(ids2.max()) < 32
    assert all(len(set(row.tolist())) == 4 for row in ids2)          # distinct experts per token
    assert len(set(ids2.reshape(-1).tolist())) > 8                    # spread over the experts
    w3, ids3 = r.select_experts(torch.zeros(10, 8, dtype=torch.bfloat16), torch.zeros(10, 32))
    assert ids3 is ids


def test_expert_load_from_both_group_list_forms():
    """Counts (type 1) and running totals (type 0) must add the same loads (routed_experts.py:571-587)."""
    import types

    import torch

    from vllm_ascend_amd.fused_moe.contracts import FusedExpertsResult
    from vllm_ascend_amd.fused_moe.layer import AscendRoutedExperts

    counts = torch.tensor([3, 0, 5, 1], dtype=torch.int64)
    for multi_stage in (False, True):
        holder = types.SimpleNamespace(
            multi_stage=multi_stage, num_iter=3, load_counter=torch.zeros((), dtype=torch.int32),
            moe_load=torch.zeros((3, 4), dtype=torch.int32) if multi_stage else torch.zeros(4, dtype=torch.int64))
        for glt, tokens in ((1, counts), (0, counts.cumsum(0)), (1, counts), (0, counts.cumsum(0))):
            res = FusedExpertsResult(routed_out=torch.zeros(1), group_list_type=glt, expert_tokens=tokens)
            AscendRoutedExperts._record_expert_load(holder, res)
        if multi_stage:
            assert holder.moe_load.tolist() == [(2 * counts).tolist(), counts.tolist(), counts.tolist()]
            assert int(holder.load_counter) == 4
        else:
            assert holder.moe_load.tolist() == (4 * counts).tolist()
    res = FusedExpertsResult(routed_out=torch.zeros(1))
    try:
        AscendRoutedExperts._record_expert_load(holder, res)
    except AssertionError as e:
        assert "should not be None when dynamic_eplb is enabled" in str(e)
    else:
        raise AssertionError("a result without expert_tokens must be refused")


def test_layer_kernel_names_follow_the_form():
    """The kernel of the routed gate_up product, as the whole-layer call launches it (no GPU: a pure function)."""
    from vllm_ascend_amd import _lib

    lib = _lib.load()

    def name(T, weights=0, hidden=2048, experts=128, inter=768, shared=0, pair_order=1):
        a = _lib.Layer(hidden=hidden, intermediate=inter, num_experts=experts, top_k=8, k_group=1, group_count=1,
                       x_dtype=_lib.DT_BF16, weights=weights, pair_order=pair_order, w13=256, s13=256, w2=256, s2=256,
                       group13=256, group2=256, shared=shared, shared_intermediate=inter, shared_alpha=1.0,
                       shared_w13=256, shared_s13=256, shared_w2=256, shared_s2=256)
        return lib.moe355_layer_kernel_name(ctypes.byref(a), T).decode()

    assert name(1) == "few_up_kernel" and name(64) == "gmm_stream_kernel"
    assert name(1, shared=1) == "few_up_kernel with the shared expert"
    big = dict(hidden=7168, experts=256, inter=2048)
    assert name(64, shared=1, **big) == "gmm_stream_kernel with the shared expert"
    assert name(64, pair_order=0, **big) == "gmm_tiled_kernel" == name(512, **big)
    assert name(4096, **big) == "gmm_wide_kernel"
    assert name(16, weights=2, **big) == "gmm_w4_pairs_kernel" and name(512, weights=2, **big) == "gmm_w4_stream_kernel"
    assert name(0) == "" and name(4, shared=3) == ""
    assert lib.moe355_layer_kernel_name(None, 4) == b""


def test_a_shared_expert_that_the_pair_order_launches_can_take_is_in_them():
    """Also where the down product could re-quantise inside instead (no GPU: a pure function).  With it the layer stays in
    pair order up to 256 MiB of repeated weight reads instead of 128."""
    from vllm_ascend_amd import _lib

    lib = _lib.load()

    def name(T, experts, hidden, inter, top_k, shared, **kw):
        args = dict(hidden=hidden, intermediate=inter, num_experts=experts, top_k=top_k, k_group=1, group_count=1,
                    x_dtype=_lib.DT_BF16, pair_order=1, w13=256, s13=256, w2=256, s2=256, shared=shared,
                    shared_intermediate=inter, shared_alpha=1.0, shared_w13=256, shared_s13=256, shared_w2=256, shared_s2=256)
        return lib.moe355_layer_kernel_name(ctypes.byref(_lib.Layer(**{**args, **kw})), T).decode()

    merged = "gmm_stream_kernel with the shared expert"
    for T in (9, 56, 57, 64, 127):
        for inter in (512, 768, 1024):
            for shared in (1, 2):
                assert name(T, 128, 2048, inter, 8, shared) == merged
                assert name(min(T, 64), 64, 2048, inter, 8, shared) == merged
            assert name(T, 128, 2048, inter, 8, 1, shared_intermediate=2 * inter) == "gmm_stream_kernel"
            assert name(T, 128, 2048, inter, 8, 1, shared_alpha=1.5) == "gmm_stream_kernel"
            assert lib.moe355_gmm2_requant_pairs_supported(T, 8, 2048, inter, 128) == (T <= 56 or inter <= 768)
    for shared in (1, 2):
        assert name(170, 8, 4096, 2048, 2, shared) == merged and name(171, 8, 4096, 2048, 2, shared) == "gmm_tiled_kernel"
    assert name(143, 8, 4096, 2048, 2, 0) == "gmm_stream_kernel" and name(144, 8, 4096, 2048, 2, 0) == "gmm_tiled_kernel"
    assert not lib.moe355_pair_order(144, 2, 8, 8, 4096, 2048) and lib.moe355_pair_order(143, 2, 8, 8, 4096, 2048)


# (experts, slots, hidden, intermediate) and the most tokens that the first launch gates and quantises by itself: the
# comparisons grow with the experts and the tokens, the rounds over a row's values with the hidden size, and more than 256 or
# 576 workgroups wait for each other
@pytest.mark.parametrize("experts, top_k, hidden, inter, most", [
    (8, 2, 1024, 1408, 3), (32, 4, 1024, 256, 4), (32, 4, 2048, 512, 2), (64, 8, 2048, 512, 2), (64, 2, 1024, 1024, 4),
    (128, 8, 2048, 768, 1), (128, 4, 2048, 768, 1), (128, 8, 512, 256, 2), (256, 8, 2048, 256, 1), (256, 4, 4096, 384, 0),
    (256, 8, 7168, 2048, 0), (1, 1, 2048, 1408, 4)])
def test_gating_inside_the_first_launch_where_it_is_short(experts, top_k, hidden, inter, most):
    from vllm_ascend_amd import _lib

    lib = _lib.load()
    a = _lib.Layer(hidden=hidden, intermediate=inter, num_experts=experts, top_k=top_k, k_group=1, group_count=1,
                   x_dtype=_lib.DT_BF16, pair_order=1, w13=256, s13=256, w2=256, s2=256)
    assert [lib.moe355_layer_gates_inside(ctypes.byref(a), T) for T in range(6)] == [int(1 <= T <= most) for T in range(6)]
    assert lib.moe355_layer_gates_inside(None, 1) == 0


def _code_objects(data):
    """Where the gfx code objects (ELF files for machine 224) inside a library start."""
    at = data.find(b"\x7fELF", 4)
    while at >= 0:
        if int.from_bytes(data[at + 18:at + 20], "little") == 224:
            yield at
        at = data.find(b"\x7fELF", at + 4)


def _kernel_metadata(path):
    """name -> metadata of every kernel of the library, from the notes of its code objects."""
    import struct

    import msgpack

    data, kernels = open(path, "rb").read(), {}
    for at in _code_objects(data):
        (sections,), (size, count) = struct.unpack_from("<Q", data, at + 40), struct.unpack_from("<2H", data, at + 58)
        for i in range(count):
            _, kind, _, _, offset, length = struct.unpack_from("<2I4Q", data, at + sections + i * size)
            if kind != 7:  # SHT_NOTE
                continue
            end, p = at + offset + length, at + offset
            while p < end:
                name, desc, note = struct.unpack_from("<3I", data, p)
                body = p + 12 + (name + 3) // 4 * 4
                if note == 32:  # NT_AMDGPU_METADATA
                    for k in msgpack.unpackb(data[body:body + desc])["amdhsa.kernels"]:
                        kernels[k[".name"]] = k
                p = body + (desc + 3) // 4 * 4
    return kernels


def test_few_token_down_product_leaves_registers_for_the_kernels_beside_it():
    """96 registers for each of its four wavefronts of a SIMD and 128 for one of the routed gate_up product are the 512 that
    there are; registers are handed out in eights."""
    from vllm_ascend_amd import _lib

    kernels = _kernel_metadata(_lib.LIB_PATH)
    down = {n: k for n, k in kernels.items() if "few_down_kernel" in n}
    beside = [k for n, k in kernels.items() if "gmm_stream_kernelILi1ELi4ELi4ELi3ELb0ELb1ELb1E" in n]
    assert len(down) == 6 and len(beside) == 1
    assert beside[0][".vgpr_count"] <= 128
    for name, k in down.items():
        assert k[".vgpr_count"] + k.get(".agpr_count", 0) <= 96, name
        assert k[".private_segment_fixed_size"] == 0, name  # nothing spilled for it


# a product that streams with workgroups for at most half of the chip (128, of 64 channels) reads its weights twice for
# nothing: tiles from 48 rows per expert instead of 32, if K is long enough for it to matter and the experts are few
@pytest.mark.parametrize("experts, k, n, first", [(8, 1024, 512, 48), (8, 960, 512, 32), (8, 4096, 1024, 48), (8, 4096, 1088, 32),
                                                  (4, 7168, 2048, 48), (4, 7168, 2112, 32), (9, 4096, 512, 32)])
def test_few_streaming_workgroups_keep_streaming(experts, k, n, first):
    from vllm_ascend_amd import _lib

    name = _lib.load().moe355_gmm_kernel_name
    for epilogue in (0, 1, 2):
        assert name(epilogue, first * experts - 1, k, n, experts) == b"gmm_stream_kernel"
        assert name(epilogue, first * experts, k, n, experts) == b"gmm_tiled_kernel"


# where the weight-streaming tiles begin, by columns of 512 channels over all experts, and by experts and K from 2048 columns on
@pytest.mark.parametrize("experts, k, n, first", [(127, 7168, 4096, 64), (128, 7168, 4096, 40), (255, 4096, 4096, 40), (256, 4096, 4096, 28),
                                                  (256, 5120, 4096, 17), (256, 5056, 4096, 28), (256, 7168, 4096, 17), (512, 4096, 2048, 28),
                                                  (256, 4032, 4096, None), (192, 7168, 5632, 28), (228, 4096, 4160, 28),
                                                  (227, 4096, 4160, 40), (128, 8192, 8192, 28), (64, 6144, 16384, 28)])
def test_where_weight_streaming_tiles_begin(experts, k, n, first):
    from vllm_ascend_amd import _lib

    name = _lib.load().moe355_gmm_kernel_name
    for epilogue in (0, 1, 2):
        for rows in (16, 17, 27, 28, 39, 40, 63, 64):
            want = "wide" if first and rows >= first else "tiled"
            assert name(epilogue, rows * experts, k, n, experts).decode() == f"gmm_{want}_kernel", rows


# above 256 rows per expert: weight-streaming tiles for weights of 32 MiB an expert, from 384 rows on (512 below 768 columns of
# tiles) of 14 MiB with at least 5120 channels, of 20 MiB with fewer, from 3072 on, at K from 5120 on with 768 columns
@pytest.mark.parametrize("experts, k, n, first", [(16, 4096, 8192, 257), (15, 4096, 8192, None), (32, 4096, 8128, 512),
                                                  (48, 4096, 8128, 384), (55, 2048, 7168, 384), (54, 2048, 7168, 512),
                                                  (64, 2048, 7104, None), (64, 3072, 5056, None), (18, 2048, 7168, None),
                                                  (19, 2048, 7168, 512), (64, 1984, 16384, None), (256, 7168, 4096, 384),
                                                  (96, 7168, 4096, 384), (95, 7168, 4096, None), (256, 5120, 4096, 384),
                                                  (256, 5120, 4032, None), (160, 5056, 4608, None), (160, 7168, 3072, 384),
                                                  (160, 7168, 3008, None)])
def test_weight_streaming_tiles_of_many_rows(experts, k, n, first):
    from vllm_ascend_amd import _lib

    name = _lib.load().moe355_gmm_kernel_name
    for epilogue in (0, 1, 2):
        for rows in (257, 383, 384, 511, 512, 2000):
            want = "wide" if first and rows >= first else "tiled"
            assert name(epilogue, rows * experts, k, n, experts).decode() == f"gmm_{want}_kernel"


# tokens of a tile in LDS: channels that fill 11 of 16 places of the wavefronts, from 1024 on; rows of fewer than 640 values only
# from 2048 channels on, 15 of 16 places (all of them below 384) and below 4096 rows; rounds of the chip that are full enough
@pytest.mark.parametrize("rows, experts, k, n, resident", [
    (65536, 128, 768, 1024, True), (65536, 128, 768, 960, False), (65535, 128, 768, 1024, False), (65536, 128, 768, 1088, False),
    (65536, 128, 768, 1280, False), (65536, 128, 768, 1344, False), (65536, 128, 768, 1408, True), (65536, 128, 768, 2112, True),
    (65536, 128, 896, 2048, True), (65536, 128, 1024, 2048, False), (65536, 128, 704, 2048, False), (65536, 128, 512, 1024, False),
    (65536, 128, 512, 1984, False), (65536, 128, 512, 2048, True), (65536, 128, 384, 2560, False), (65536, 128, 384, 2880, True),
    (65536, 128, 256, 2880, False), (65536, 128, 256, 4096, True), (65536, 16, 512, 2048, False), (65520, 16, 512, 2048, True),
    (65536, 16, 640, 2048, True), (128 * 288 - 1, 128, 768, 2048, False), (128 * 288, 128, 768, 2048, True),
    (34000, 8, 640, 2048, False), (37759, 8, 640, 2048, False), (37760, 8, 640, 2048, False), (37888, 8, 640, 2048, True),
    (48640, 8, 640, 2048, True), (48768, 8, 640, 2048, False), (50688, 8, 640, 2048, True), (40000, 1, 640, 2048, False)])
def test_tokens_of_a_tile_in_lds_lines(rows, experts, k, n, resident):
    from vllm_ascend_amd import _lib

    name = _lib.load().moe355_gmm_kernel_name
    assert (name(2, rows, k, n, experts) == b"gmm_resident_kernel") == resident
    assert name(0, rows, k, n, experts) != b"gmm_resident_kernel" != name(1, rows, k, n, experts)


# where the column workgroups of a gate_up tile exchange the rows' maxima: rows of their tiles
@pytest.mark.parametrize("experts, k, n, rows, tile_rows", [
    (256, 7168, 4096, 4096, 128), (256, 7168, 4096, 256 * 144, 256), (256, 7168, 4096, 256 * 145, 0), (128, 2048, 2048, 1152, 128),
    (128, 2048, 1536, 1024, 64), (128, 2048, 1536, 128 * 64 - 1, 64), (128, 2048, 1536, 128 * 64, 128), (128, 2048, 1536, 65536, 128),
    (256, 2048, 1536, 256 * 48 - 1, 0), (256, 2048, 1536, 256 * 48, 128), (64, 4096, 3072, 1152, 0), (128, 4096, 3072, 10240, 0),
    (32, 2880, 5760, 9600, 0), (8, 1024, 2816, 1040, 64), (8, 1024, 2816, 16000, 128), (128, 2048, 1536, 512, 0), (1, 2048, 4096, 4096, 0),
    (128, 2048, 1536, 65544, 0), (128, 2048, 1536, 100000, 0), (512, 1024, 2048, 20000, 128), (513, 1024, 2048, 20000, 0)])
def test_where_gate_up_tiles_quantise_their_rows(experts, k, n, rows, tile_rows):
    from vllm_ascend_amd import _lib

    assert _lib.load().moe355_meeting_tile_rows(rows, k, n, experts) == tile_rows


def test_columns_of_a_routed_tile_have_places():
    """96 workgroups of the 64-row tiles run on an XCD, 64 of the 128-row ones and 32 of the wide ones, where a tall tile may wait with
    both halves; a launch may hold all but one of a tile's columns, and another stream's launch as many."""
    from vllm_ascend_amd import _lib

    rows_of = _lib.load().moe355_meeting_tile_rows
    seen = set()
    for experts in (1, 4, 6, 10, 16, 32, 128, 256, 512):
        for k in (64, 384, 1024, 2880, 7168):
            for n in [*range(64, 12289, 192), *range(12288, 50000, 512)]:
                for rows in (6, 18, 48, 63, 100, 144, 250, 1000):
                    tile = rows_of(rows * experts, k, n, experts)
                    seen.add(tile)
                    assert -(-n // (512 if tile == 256 else 256)) <= {0: n, 64: 48, 128: 16, 256: 8}[tile], (experts, k, n, rows)
    assert seen == {0, 64, 128, 256}


def test_no_words_for_a_meeting_that_does_not_take_place():
    """The words (a word for every pair and column of a tile) end with the one-launch map, at 65536 pairs."""
    from vllm_ascend_amd import _lib

    lib = _lib.load()

    def workspace(tokens, weights, shared=0):
        a = _lib.Layer(hidden=2048, intermediate=768, num_experts=128, top_k=8, k_group=1, group_count=1, weights=weights,
                       x_dtype=_lib.DT_BF16, w13=256, s13=256, w2=256, s2=256, group13=256, group2=256, shared=shared,
                       shared_intermediate=1024, shared_alpha=1.0, shared_w13=256, shared_s13=256, shared_w2=256, shared_s2=256)
        return lib.moe355_layer_workspace(ctypes.byref(a), tokens)

    assert lib.moe355_meeting_tile_rows(65536, 2048, 1536, 128) == 128  # six columns
    assert lib.moe355_shared_meeting_columns(8192, 2048, 2048, None) == 8  # a word for every pair
    for weights, shared, words in ((0, 0, 6), (0, 1, 7), (2, 0, 0), (2, 1, 1)):
        # what one token more adds, above 8192 and there
        step = [workspace(t + 1, weights, shared) - workspace(t, weights, shared) for t in (8191, 8192, 8193, 8194)]
        usual = max(abs(s) for s in (step[0], step[2], step[3]))
        assert usual < 1 << 17
        assert abs(step[1] + words * 65536 * 4) < 1 << 18, (weights, shared, step)


# ... and of the shared expert's: all columns of a row of tiles that fall to one XCD have a place there, also beside such a launch on
# another stream (32 workgroups of 160 KiB of LDS run on one; each launch may hold all but one of a row's columns)
def test_columns_that_meet_have_places():
    from vllm_ascend_amd import _lib

    lib, on_one = _lib.load(), ctypes.c_int()
    admitted = 0
    for n in (512, 1408, 4096, 4224, 5632, 8192, 8256, 10240, 11264, 16256, 16384):
        for rows in [*range(1, 65537, 255), 32000, 40192, 44288, 64768, 65536]:
            columns = lib.moe355_shared_meeting_columns(rows, 64, n, ctypes.byref(on_one))
            want = -(-n // 256) if -(-rows // 256) * -(-n // 256) >= 192 else 0
            assert columns == want
            assert (0 < on_one.value <= min(16, columns)) if columns else on_one.value == 0
            assert 8 * on_one.value >= columns
            admitted += columns > 16 and rows > 30000
    assert admitted > 100
    assert lib.moe355_shared_meeting_columns(65536, 64, 16384 + 64, ctypes.byref(on_one)) == 0  # 65 columns
    assert lib.moe355_shared_meeting_columns(0, 64, 4096, None) == 0 == lib.moe355_shared_meeting_columns(4096, 64, 0, None)


def test_looks_of_the_next_call_are_bounded():
    """moe355::take_meeting_looks() is what a layer call takes; it has no C name."""
    from vllm_ascend_amd import _lib

    lib = _lib.load()
    taken = lib._ZN6moe35518take_meeting_looksEv
    usual = taken()
    assert usual == 4096
    for looks, want in ((0, 0), (1, 1), (4095, 4095), (4096, 4096), (4097, 4096), (2**31 - 1, 4096)):
        assert lib.moe355_next_meeting_looks(looks) == 0
        assert taken() == want and taken() == usual
    assert lib.moe355_next_meeting_looks(-1) == -1 and taken() == usual


# one for every 56 pairs, but not where a short launch (fewer than 1536 units of 64 channels) has places in front of its slots
# (from two pairs per expert on), nor from twelve pairs per expert on
@pytest.mark.parametrize("experts, n, pairs, blocks", [(128, 1536, 512, 9), (128, 512, 256, 4), (128, 512, 257, 0), (128, 704, 512, 0),
                                                       (128, 768, 512, 9), (64, 1024, 512, 0), (256, 512, 512, 9),
                                                       (128, 1536, 33, 0), (60, 2816, 719, 12), (60, 2816, 720, 0),
                                                       (128, 4096, 383, 0), (128, 4096, 384, 6)])
def test_further_blocks_in_front_of_the_slots(experts, n, pairs, blocks):
    from vllm_ascend_amd import _lib

    assert _lib.load().moe355_pair_blocks_in_front(pairs, n, experts) == blocks


# the re-quantisation inside the down product: three and a half pairs per expert, eight with short rows if the hot experts'
# rows are not taken in passes
@pytest.mark.parametrize("experts, top_k, n, k, most", [(32, 4, 4096, 768, 28), (64, 6, 4096, 640, (37, 64, 85)), (64, 8, 2048, 768, 64),
                                                        (64, 8, 2048, 800, 28), (128, 8, 2048, 768, 128), (128, 8, 6144, 256, 56),
                                                        (128, 8, 4096, 256, 128)])
def test_re_quantisation_inside_the_down_product(experts, top_k, n, k, most):
    from vllm_ascend_amd import _lib

    supported = _lib.load().moe355_gmm2_requant_pairs_supported
    first, again, last = most if isinstance(most, tuple) else (most, most, most)
    for T in range(1, 1024 // top_k + 1):
        assert bool(supported(T, top_k, n, k, experts)) == (T <= first or again <= T <= last), T
