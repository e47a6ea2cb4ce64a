"""The gate_up product whose tiles' workgroups exchange the maxima of their rows and store int8, against the operators (fp32
values in memory, a launch that quantises them): the same bits, also where a workgroup gives up looking for the others'."""
import dataclasses

import pytest
import torch

from _inputs import CONFIGS, make_layer
from _layer_utils import build_layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _lib():
    from vllm_ascend_amd._lib import load

    return load()


def _layer(tokens, **shape):
    cfg = dataclasses.replace(CONFIGS["c2_small"], T=tokens, **shape)
    d = make_layer(cfg, seed=tokens)
    return cfg, build_layer(cfg, d, DEV), d["x"].to(DEV), d["logits"].to(DEV)


def _random_layer(tokens, E, k, H, I):
    """Weights made on the GPU: the shapes that reach the weight-streaming tiles are too large for the host's generator."""
    cfg = dataclasses.replace(CONFIGS["c2_small"], T=8, E=E, k=k, H=64, I=32)
    d = make_layer(cfg, seed=tokens)
    g = torch.Generator(device=DEV).manual_seed(tokens)
    for name, shape in (("w13", (E, 2 * I, H)), ("w2", (E, H, I))):
        d[name] = torch.randint(-128, 128, shape, generator=g, device=DEV, dtype=torch.int8)
    d["s13"], d["s2"] = (torch.rand(E, n, generator=g, device=DEV) * 0.009 + 0.001 for n in (2 * I, H))
    layer = build_layer(dataclasses.replace(cfg, T=tokens, H=H, I=I), d, DEV)
    x = torch.randn(tokens, H, generator=g, device=DEV).to(torch.bfloat16)
    return layer, x, torch.randn(tokens, E, generator=g, device=DEV)


def _tile_rows(layer, T):
    """Rows of the tiles whose workgroups meet in a call of T tokens, 0 where they do not.  (The layer has been called before.)"""
    plan = layer._layer_plan
    a = plan.desc
    if _lib().moe355_layer_kernel_name(plan.ref, T) not in (b"gmm_tiled_kernel", b"gmm_wide_kernel"):
        return 0
    return _lib().moe355_meeting_tile_rows(T * a.top_k, a.hidden, 2 * a.intermediate, a.num_experts)


def _check(layer, x, logits, looks=(None,), tile_rows=(64, 128, 256)):
    """tile_rows: of the routed experts' tiles, any of which the case is meant for."""
    want = layer.forward_impl(x, logits).routed_out
    for n in looks:
        if n is not None:
            assert _lib().moe355_next_meeting_looks(n) == 0
        got = layer(x, logits)
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), n
    assert _tile_rows(layer, x.shape[0]) in tile_rows


def _with_shared(layer, S, H, seed, overlap=False, limit=0.0):
    from vllm_ascend_amd.fused_moe.shared_experts import AscendSharedExperts

    g = torch.Generator(device=DEV).manual_seed(seed)
    up, down = (torch.randint(-128, 128, shape, generator=g, device=DEV, dtype=torch.int8) for shape in ((2 * S, H), (H, S)))
    up_scale, down_scale = (torch.rand(n, generator=g, device=DEV) * 0.009 + 0.001 for n in (2 * S, H))
    layer.shared_experts = AscendSharedExperts(up, up_scale, down, down_scale, multistream_overlap=overlap, swiglu_limit=limit)


# one column block and several, whole and partial ones (128 values each; 40 and 47 of the 48 that there may be), 64- and 128-row tiles,
# a list whose tiles two XCDs share, K of one step and of every remainder modulo the ring
@pytest.mark.parametrize("E, k, T, H, I, tile_rows", [
    (8, 2, 512, 64, 32, 128), (8, 2, 513, 128, 160, 128), (8, 2, 515, 192, 288, 64), (8, 2, 521, 256, 512, 64), (6, 2, 600, 320, 1408, 64),
    (32, 4, 517, 512, 512, 64), (16, 4, 2049, 256, 1024, 128), (64, 8, 384, 448, 640, 128), (128, 8, 257, 256, 640, 64),
    (96, 8, 257, 256, 1024, 128), (16, 2, 500, 384, 5120, 64), (16, 4, 250, 320, 5984, 64)])
@pytest.mark.parametrize("skew", [0.0, 3.0])
def test_layers_on_tiles(E, k, T, H, I, tile_rows, skew):
    print(f"E={E} k={k} T={T} H={H} I={I} skew={skew} tiles of {_lib().moe355_meeting_tile_rows(T * k, H, 2 * I, E)}", flush=True)
    cfg, layer, x, logits = _layer(T, E=E, k=k, H=H, I=I)
    logits = logits - skew * torch.arange(E, device=DEV).float().log1p()
    _check(layer, x, logits, looks=(None, 0, 1), tile_rows=(tile_rows,))


# rows at the edges of a tile and of a wavefront's groups of 16
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 192, 193])
def test_rows_of_an_expert(rows):
    T, E = 1024, 8
    cfg, layer, x, logits = _layer(T, E=E, k=1, H=128, I=256)
    logits = torch.full((T, E), -9.0, device=DEV)
    logits[torch.arange(T), torch.where(torch.arange(T) < rows, 0, 1 + torch.arange(T) % (E - 1))] = 9.0
    _check(layer, x, logits, looks=(None, 0))


@pytest.mark.parametrize("limit", [0.0, 0.7])
def test_clamp_infinities_and_zeros(limit):
    cfg, layer, x, logits = _layer(640, E=8, k=2, H=256, I=512)
    layer.moe_config = dataclasses.replace(layer.moe_config, swiglu_limit=limit)
    x = x.clone()
    x[3] = 0
    x[70] = float("inf")
    x[200, 5] = float("nan")
    x[300] *= 1e30
    _check(layer, x, logits, looks=(None, 0))


# weight-streaming tiles: one to six blocks of 32 rows, tall ones with an entry for every half and with one for both, alone and
# beside short ones; the last column block of 512 channels a half one, an odd number of them
@pytest.mark.parametrize("E, k, H, I, T, skew", [
    (64, 8, 1024, 1024, 1000, 0.0), (64, 8, 1024, 1024, 1100, 0.3), (64, 8, 1024, 1024, 1100, 1.1), (128, 8, 1024, 640, 2000, 0.0),
    (128, 8, 1024, 640, 1900, 1.1), (128, 8, 1088, 672, 2000, 0.5), (16, 2, 1024, 256, 1000, 0.2)])
def test_layers_on_weight_streaming_tiles(E, k, H, I, T, skew):
    print(f"E={E} k={k} T={T} H={H} I={I} skew={skew}", flush=True)
    layer, x, logits = _random_layer(T, E, k, H, I)
    _check(layer, x, logits - skew * torch.arange(E, device=DEV).float().log1p(), looks=(None, 0), tile_rows=(256,))


def _ms(layer, x, logits, looks):
    """The fastest of five calls."""
    best = float("inf")
    for _ in range(5):
        if looks is not None:
            assert _lib().moe355_next_meeting_looks(looks) == 0
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        layer(x, logits)
        end.record()
        torch.cuda.synchronize()
        best = min(best, start.elapsed_time(end))
    return best


# A workgroup that gives up computes a column's maxima by one scalar product after the other, some ten times as long as the whole
# product takes.  After one look in vain it computes the first column that is missing, if that has not come meanwhile; the words of
# the others come while it does.  Without a look it computes seven of the eight (0.05 and 4.8 ms a call).
def test_columns_that_have_come_are_not_computed():
    T, E, H, I = 1024, 8, 2048, 1024
    cfg, layer, x, logits = _layer(T, E=E, k=1, H=H, I=I)
    layer(x, logits)
    assert _tile_rows(layer, T) and I // 128 == 8
    one, all_of_them = _ms(layer, x, logits, 1), _ms(layer, x, logits, 0)
    print(f"one look {one:.3f} ms, none {all_of_them:.3f} ms", flush=True)
    assert one < 0.5 * all_of_them


# The results are the same where nobody meets: what shows it is the time.  A call whose workgroups compute everybody's maxima takes
# ten times as long as one whose workgroups meet; one whose workgroups wait in vain would take longer still.
@pytest.mark.parametrize("E, k, T, H, I, tile_rows", [(128, 8, 288, 2048, 768, 64), (64, 8, 500, 2048, 1024, 128),
                                                      (64, 8, 1000, 1024, 1024, 256)])
def test_workgroups_meet(E, k, T, H, I, tile_rows):
    layer, x, logits = _random_layer(T, E, k, H, I)
    _check(layer, x, logits, looks=(None, 0), tile_rows=(tile_rows,))
    usual, alone = _ms(layer, x, logits, None), _ms(layer, x, logits, 0)
    print(f"E={E} T={T} H={H} I={I}: {usual:.3f} ms, {alone:.3f} ms without a look", flush=True)
    assert usual < 0.5 * alone


# 17 columns of a row of tiles would fall to an XCD if only the perimeter of its rectangle counted, and 64 of them in three rows
@pytest.mark.parametrize("T, S, columns", [(8192, 4224, 33), (700, 8192, 64)])
def test_workgroups_of_the_shared_expert_meet(T, S, columns):
    H = 256
    assert _lib().moe355_shared_meeting_columns(T, H, 2 * S, None) == columns
    cfg, layer, x, logits = _layer(T, E=8, k=2, H=H, I=64)
    _with_shared(layer, S, H, T)
    _check(layer, x, logits, looks=(None, 0), tile_rows=(0, 64, 128, 256))
    usual, alone = _ms(layer, x, logits, None), _ms(layer, x, logits, 0)
    print(f"T={T} S={S}: {usual:.3f} ms, {alone:.3f} ms without a look", flush=True)
    assert usual < 0.5 * alone


# workgroups of another launch hold places of those that are waited for
@pytest.mark.parametrize("T, I, S", [(3072, 512, 2048), (3072, 512, 512), (600, 1408, 1408)])
def test_beside_a_shared_expert_on_its_side_stream(T, I, S):
    H = 512
    cfg, layer, x, logits = _layer(T, E=8, k=2, H=H, I=I)
    _with_shared(layer, S, H, T, overlap=True)
    _check(layer, x, logits, looks=(None, None, 1, 0))
    assert layer._layer_plan.desc.shared == 2


@pytest.mark.parametrize("S", [0, 2048])
def test_captured_and_from_two_streams(S):
    T = 3072 if S else 700
    cfg, layer, x, logits = _layer(T, E=8, k=2, H=256, I=640)
    if S:
        assert _lib().moe355_shared_meeting_columns(T, 256, 2 * S, None) == 16
        _with_shared(layer, S, 256, T)
    want = layer.forward_impl(x, logits).routed_out
    layer(x, logits)
    torch.cuda.synchronize()
    assert _tile_rows(layer, T)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer(x, logits)
    side = torch.cuda.Stream()
    for _ in range(5):
        out.zero_()
        graph.replay()
        with torch.cuda.stream(side):
            beside = [layer(x, logits) for _ in range(3)]
        torch.cuda.synchronize()
        assert torch.equal(out, want) and all(torch.equal(b, want) for b in beside)


# the shared expert of a prefill batch, 256 x 256 tiles: whole and partial row tiles and column blocks, one round of workgroups
# and several, as many columns as meet and one more, words of the meeting that do and do not fill whole rows of the routed experts' pairs, beside int4 experts
@pytest.mark.parametrize("T, S, H, k, w4", [
    (3072, 2048, 64, 2, False), (3007, 2016, 192, 3, False), (12200, 512, 128, 1, False), (6001, 1984, 256, 8, False), (3009, 2048, 128, 2, True),
    (700, 8192, 64, 2, False), (700, 8224, 64, 2, False)])
@pytest.mark.parametrize("limit", [0.0, 0.7])
def test_shared_expert_on_dense_tiles(T, S, H, k, w4, limit):
    print(f"T={T} S={S} H={H} k={k} w4={w4} limit={limit}", flush=True)
    assert -(-T // 256) * -(-2 * S // 256) >= 192
    assert _lib().moe355_shared_meeting_columns(T, H, 2 * S, None) == (-(-S // 128) if S <= 8192 else 0)
    cfg = dataclasses.replace(CONFIGS["c5_small_perchannel" if w4 else "c2_small"], T=T, E=8, k=k, H=H, I=64)
    d = make_layer(cfg, seed=T)
    layer = build_layer(cfg, d, DEV)
    _with_shared(layer, S, H, T, limit=limit)
    x = d["x"].to(DEV).clone()
    x[3] = 0
    x[70] = float("inf")
    x[300] *= 1e30
    _check(layer, x, d["logits"].to(DEV), looks=(None, 0, 1), tile_rows=(0, 64, 128, 256))
