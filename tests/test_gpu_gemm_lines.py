"""The GEMMs on both sides of the lines between their families: streaming and the tiles at 1023 / 1024 rows for a small product,
fewer rows than experts / one row per expert for one of a GiB and more, 63 / 64 rows per expert at a long K."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def exact_products(x, w, counts):
    """The int32 sums of the experts' rows, by torch in 64-bit floating point (exact: they are whole and below 2^53)."""
    out, row = [], 0
    for e, m in enumerate(counts.tolist()):
        out.append((x[row:row + m].double() @ w[e].double().t().contiguous()).int())
        row += m
    return torch.cat(out)


LINES = [(1023, 128, 256, 128, "stream"), (1024, 128, 256, 128, "tiled"), (1100, 1200, 64, 64, "stream"),
         (63 * 8 + 7, 8, 4096, 128, "tiled"), (64 * 8, 8, 4096, 128, "wide"),
         (287, 288, 2048, 2048, "stream"), (288, 288, 2048, 2048, "tiled"),
         (255, 256, 2048, 2048, "stream"), (256, 256, 2048, 2048, "tiled"), (256 * 23, 256, 4096, 1024, "tiled")]


@pytest.mark.parametrize("skewed", [False, True])
@pytest.mark.parametrize("R,E,Kd,N,family", LINES)
def test_families_on_both_sides_of_a_line(R, E, Kd, N, family, skewed):
    from oracle import oracle as orc
    from vllm_ascend_amd import kernels as K
    from vllm_ascend_amd._lib import W_ENK, load

    print(f"line R={R} E={E} K={Kd} N={N} {family} skewed={skewed}", flush=True)
    assert load().moe355_gmm_kernel_name(2, R, Kd, N, E).decode() == f"gmm_{family}_kernel"
    rng = np.random.default_rng(R + E)
    p = 1.0 / (rng.permutation(E) + 1.0) ** (1.1 if skewed else 0.0)
    cum = torch.from_numpy(np.cumsum(rng.multinomial(R, p / p.sum())).astype(np.int64))
    g = torch.Generator().manual_seed(R)
    x = torch.randint(-128, 128, (R, Kd), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (E, N, Kd), generator=g, dtype=torch.int8)
    sw = torch.rand(E, N, generator=g) * 0.009 + 0.001
    sx = torch.rand(R, generator=g) * 0.05 + 0.001
    wnz = K.format_cast_nz(w.to("cuda"), W_ENK)
    ref = orc.gmm_i32(x.numpy(), w.numpy(), cum.numpy())
    got = K.gmm2_dequant(x.to("cuda"), wnz, sw.to("cuda"), sx.to("cuda"), cum.to("cuda"), 0, N, Kd)
    torch.cuda.synchronize()
    want = orc.gmm2_dequant(ref, sx.numpy(), sw.numpy(), cum.numpy())
    assert np.array_equal(got.cpu().contiguous().view(torch.int16).numpy().view(np.uint16), want)
    q_want, s_want = orc.swiglu_quant(orc.dequant_acc(ref, sx.numpy(), sw.numpy(), cum.numpy()))
    q, s = K.gmm1_swiglu_quant(x.to("cuda"), wnz, sw.to("cuda"), sx.to("cuda"), cum.to("cuda"), 0, N, Kd)
    torch.cuda.synchronize()
    assert np.array_equal(q.cpu().numpy(), q_want)
    assert np.array_equal(s.cpu().numpy().view(np.uint32), s_want.view(np.uint32))


# rows of the down GEMM that re-quantises: shorter than, equal to and longer than the 256 values of one load, with a
# remainder; an expert with two passes of 32 rows
@pytest.mark.parametrize("T,E,I", [(56, 128, 320), (56, 128, 256), (56, 128, 32), (40, 128, 1408), (1, 128, 1504)])
def test_requantising_down_gemm_gives_the_separate_launches_bits(T, E, I):
    from vllm_ascend_amd import kernels as K
    from vllm_ascend_amd._lib import W_ENK

    H, k = 1024, 8
    print(f"requant T={T} E={E} I={I}", flush=True)
    assert K.gmm2_requant_pairs_supported(T, k, H, I, E)
    g = torch.Generator().manual_seed(T + I)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to("cuda")
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32)
    ids[:, 0] = 5
    ids = ids.to("cuda")
    w13 = torch.randint(-128, 128, (E, 2 * I, H), generator=g, dtype=torch.int8).to("cuda")
    w2 = torch.randint(-128, 128, (E, H, I), generator=g, dtype=torch.int8).to("cuda")
    s13 = (torch.rand(E, 2 * I, generator=g) * 0.009 + 0.001).to("cuda")
    s2 = (torch.rand(E, H, generator=g) * 0.009 + 0.001).to("cuda")
    w13, w2 = K.format_cast_nz(w13, W_ENK), K.format_cast_nz(w2, W_ENK)
    xq, xs = K.dynamic_quant(x)
    q1, s1 = K.gmm1_swiglu_quant_pairs(xq, xs, ids, w13, s13, 2 * I, H)
    want = K.gmm2_dequant_pairs(q1, w2, s2, s1, ids, H, I)
    y = K.gmm1_swiglu_pairs(xq, xs, ids, w13, s13, 2 * I, H)
    got = K.gmm2_requant_dequant_pairs(y, w2, s2, ids, H, I)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


# ... y is a caller's: the maximum of a row passes over its NaNs, quiet and signalling, in each of the four places of a load and
# on either side of the row's largest value
@pytest.mark.parametrize("bits", [0x7fc00000, 0x7f800001, 0xffa00000], ids=["quiet", "signalling", "negative"])
@pytest.mark.parametrize("I", [64, 768, 1500 // 32 * 32])
def test_nan_beside_a_row_s_largest_value(I, bits):
    from vllm_ascend_amd import kernels as K
    from vllm_ascend_amd._lib import W_ENK

    T, k, E, H = 8, 4, 128, 1024
    print(f"nan in y I={I} {bits:#x}", flush=True)
    assert K.gmm2_requant_pairs_supported(T, k, H, I, E)
    g = torch.Generator().manual_seed(I)
    y = torch.randn(T * k, I, generator=g)
    for r in range(T * k):  # the largest value in place r % 4 of a load, a NaN in r / 4 % 4, one load apart in the last rows
        at = (r * 20 + 4 * (r // 8)) % (I - 8) // 4 * 4
        y[r, at + r % 4] = 50.0 + r
        y.view(torch.int32)[r, at + r // 4 % 4 + (4 if r >= 16 or r % 4 == r // 4 % 4 else 0)] = bits - (bits >> 31 << 32)
    known = torch.where(y.isnan(), 0.0, y).abs().amax(1)
    scale = known / 127.0
    q = torch.where(y.isnan(), 0.0, (y * (1.0 / scale)[:, None]).round().clamp(-128, 127)).to(torch.int8)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to("cuda")
    w2 = K.format_cast_nz(torch.randint(-128, 128, (E, H, I), generator=g, dtype=torch.int8).to("cuda"), W_ENK)
    s2 = (torch.rand(E, H, generator=g) * 0.009 + 0.001).to("cuda")
    want = K.gmm2_dequant_pairs(q.to("cuda"), w2, s2, scale.to("cuda"), ids, H, I)
    got = K.gmm2_requant_dequant_pairs(y.to("cuda"), w2, s2, ids, H, I)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


# token quantisation with a row per wavefront: from 512 tokens on, rows of up to 2048 values, a last workgroup that is
# not full
@pytest.mark.parametrize("T,H", [(511, 2048), (512, 2048), (515, 1032), (513, 8), (777, 2056)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_token_rows_quantised_beside_the_gating(T, H, dtype):
    from vllm_ascend_amd import kernels as K

    print(f"gate_quant T={T} H={H} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn(T, H, generator=g).to(dtype)
    x[3] = 0
    x[-1] *= 1e-6
    x, logits = x.to("cuda"), torch.randn(T, 128, generator=g).to("cuda")
    got = K.gate_quant(x, logits, 8, 1, 1, 0, 1, 0, 1.0, 1e-20, None)
    xq, xs = K.dynamic_quant(x)
    torch.cuda.synchronize()
    assert torch.equal(got[2], xq) and torch.equal(got[3].view(torch.int32), xs.view(torch.int32))

# A dense product (one expert) on both sides of the lines around the tiles that cut K over their wavefronts: 64 / 65 rows, as
# many 128-row tiles as half the compute units, a last tile of one row, a last row of tiles of one and of 64; more K steps
# than wavefronts, fewer (a wavefront without any), and numbers of them that leave every remainder of the register ring
SPLIT_LINES = [(64, 256, 256, "stream"), (65, 256, 256, "split"), (128, 64, 64, "split"), (129, 192, 576, "split"),
               (200, 1408, 320, "split"), (191, 832, 128, "split"), (1000, 512, 3840, "split"), (1024, 128, 4096, "tiled")]


@pytest.mark.parametrize("R,Kd,N,family", SPLIT_LINES)
def test_dense_product_with_k_cut_over_the_wavefronts(R, Kd, N, family):
    from oracle import oracle as orc
    from vllm_ascend_amd import kernels as K
    from vllm_ascend_amd._lib import W_ENK, load

    print(f"dense line R={R} K={Kd} N={N} {family}", flush=True)
    assert load().moe355_gmm_kernel_name(2, R, Kd, N, 1).decode() == f"gmm_{family}_kernel"
    g = torch.Generator().manual_seed(R)
    x = torch.randint(-128, 128, (R, Kd), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (1, N, Kd), generator=g, dtype=torch.int8)
    sw = torch.rand(1, N, generator=g) * 0.009 + 0.001
    sx = torch.rand(R, generator=g) * 0.05 + 0.001
    wnz = K.format_cast_nz(w.to("cuda"), W_ENK)
    for rows in (R, R - 1, R // 2):  # the group may hold fewer rows than the buffer
        cum = torch.tensor([rows], dtype=torch.int64)
        ref = orc.gmm_i32(x.numpy(), w.numpy(), cum.numpy())
        acc = K.gmm_i32(x.to("cuda"), wnz, cum.to("cuda"), 0, N, Kd)
        got = K.gmm2_dequant(x.to("cuda"), wnz, sw.to("cuda"), sx.to("cuda"), cum.to("cuda"), 0, N, Kd)
        q, s = K.gmm1_swiglu_quant(x.to("cuda"), wnz, sw.to("cuda"), sx.to("cuda"), cum.to("cuda"), 0, N, Kd)
        torch.cuda.synchronize()
        assert np.array_equal(acc.cpu().numpy()[:rows], ref[:rows])
        want = orc.gmm2_dequant(ref, sx.numpy(), sw.numpy(), cum.numpy())
        assert np.array_equal(got.cpu().contiguous().view(torch.int16).numpy().view(np.uint16)[:rows], want[:rows])
        q_want, s_want = orc.swiglu_quant(orc.dequant_acc(ref, sx.numpy(), sw.numpy(), cum.numpy()))
        assert np.array_equal(q.cpu().numpy()[:rows], q_want[:rows])
        assert np.array_equal(s.cpu().numpy().view(np.uint32)[:rows], s_want.view(np.uint32)[:rows])


# ... narrow products: up to 768 workgroups in rows of eight, 1024 if K is short
@pytest.mark.parametrize("R,Kd,N,family", [(6144, 1088, 64, "split"), (6145, 1088, 64, "tiled"), (3072, 1088, 576, "split"),
                                           (3073, 1088, 576, "tiled"), (8192, 64, 64, "split"), (8193, 64, 64, "tiled"),
                                           (4096, 128, 576, "split"), (4097, 128, 576, "tiled")])
def test_narrow_dense_products_with_many_rows(R, Kd, N, family):
    test_dense_product_with_k_cut_over_the_wavefronts(R, Kd, N, family)


# ... whose rows are gathered from tokens beyond 4 GiB (and, by turns, from tokens in front of them)
def test_dense_product_gathers_beyond_4_gib():
    from vllm_ascend_amd import kernels as K
    from vllm_ascend_amd._lib import W_ENK, load

    R, Kd, N = 70, 1 << 16, 128
    T = (1 << 32) // Kd + R
    print(f"dense gather R={R} K={Kd} N={N} from {T} tokens", flush=True)
    assert load().moe355_gmm_kernel_name(1, R, Kd, N, 1).decode() == "gmm_split_kernel"
    g = torch.Generator(device="cuda").manual_seed(R)
    x = torch.zeros(T, Kd, dtype=torch.int8, device="cuda")
    x[:R], x[-R:] = (torch.randint(-128, 128, (R, Kd), generator=g, dtype=torch.int8, device="cuda") for _ in range(2))
    rows = torch.arange(R, dtype=torch.int32, device="cuda")
    rows[::2] += T - R
    wnz = K.format_cast_nz(torch.randint(-128, 128, (1, N, Kd), generator=g, dtype=torch.int8, device="cuda"), W_ENK)
    sw = torch.rand(1, N, generator=g, device="cuda") * 0.009 + 0.001
    sx = torch.rand(T, generator=g, device="cuda") * 0.05 + 0.001
    cum = torch.tensor([R], dtype=torch.int64, device="cuda")
    q, s = K.gmm1_swiglu_quant_gather(x, sx, rows, wnz, sw, cum, 0, N, Kd)
    at = rows.long()
    q_want, s_want = K.gmm1_swiglu_quant(x[at], wnz, sw, sx[at], cum, 0, N, Kd)
    torch.cuda.synchronize()
    assert torch.equal(q, q_want) and torch.equal(s.view(torch.int32), s_want.view(torch.int32))


# few experts: 64-row tiles as long as they do not outnumber the compute units, and 128-row tiles
@pytest.mark.parametrize("R,E,Kd,N", [(1024, 8, 192, 1024), (3904, 8, 64, 1024), (3968, 8, 64, 1024), (1030, 3, 128, 2816)])
def test_tiles_of_half_the_height_for_few_experts(R, E, Kd, N):
    test_families_on_both_sides_of_a_line(R, E, Kd, N, "tiled", True)


# ... the last row of the line and the first one behind it: half a tile for the last one of up to 16 experts, three quarters
# of more
@pytest.mark.parametrize("E,R,Kd,N", [(8, 3903, 64, 1024), (16, 3647, 64, 1024), (17, 3391, 64, 1024), (24, 959, 64, 2048)])
def test_half_the_height_up_to_a_full_chip(E, R, Kd, N):
    from vllm_ascend_amd._lib import load

    height = load().moe355_gmm_tile_rows
    assert height(R, Kd, N, E) == 64 and height(R + 1, Kd, N, E) == 128
    for rows in (R, R + 1):
        test_families_on_both_sides_of_a_line(rows, E, Kd, N, "tiled", True)


# ... with three, two and one row at a time in a wavefront's registers: on both sides of 768 and of 1024 values, a last load
# that is not full, up to eight rows per expert, an expert with a row of every token (several passes of 32 rows)
@pytest.mark.parametrize("T,E,I", [(128, 128, 768), (128, 128, 736), (33, 128, 544), (56, 128, 800), (56, 128, 1024), (56, 128, 1056)])
def test_rows_re_quantised_several_at_a_time(T, E, I):
    test_requantising_down_gemm_gives_the_separate_launches_bits(T, E, I)


# fewer than 1024 rows: 31 / 32 rows per expert
@pytest.mark.parametrize("R,family", [(32 * 16 - 1, "stream"), (32 * 16, "tiled")])
def test_few_rows_on_tiles(R, family):
    test_families_on_both_sides_of_a_line(R, 16, 192, 320, family, True)


# ... and 47 / 48 where few experts stream with workgroups for half of the chip at most
@pytest.mark.parametrize("R,family", [(48 * 8 - 1, "stream"), (48 * 8, "tiled")])
def test_few_rows_on_tiles_few_channels(R, family):
    test_families_on_both_sides_of_a_line(R, 8, 1024, 512, family, True)


# 64 rows per expert at a long K: as many columns of wide tiles as half of the compute units, and one less
@pytest.mark.parametrize("E,family", [(63, "tiled"), (64, "wide")])
def test_columns_of_wide_tiles(E, family):
    test_families_on_both_sides_of_a_line(64 * E, E, 4096, 576, family, True)


# The down product with a tile's tokens in LDS: from 288 rows per expert and 512 workgroups of 128 rows x 1024 channels on, rows
# of 256 to 896 values in steps of 128; experts of no row, of one, at the borders of half and whole tiles; channels that leave
# every wavefront two groups of 64 (9216, 4096), some of them one (14400, 17408, 1472, whose last part is a group shorter), and
# seven of the last part none (15424)
@pytest.mark.parametrize("avg,E,Kd,N,family", [(287, 16, 384, 14400, "tiled"), (288, 16, 384, 14400, "resident"),
                                               (512, 15, 384, 9216, "resident"), (400, 12, 896, 14400, "resident"),
                                               (340, 12, 768, 17408, "resident"), (340, 12, 1024, 17408, "tiled"),
                                               (340, 12, 704, 17408, "tiled"), (340, 12, 768, 16384, "tiled"),
                                               (11000, 2, 256, 2112, "tiled"), (13000, 2, 768, 2112, "resident"),
                                               (1200, 16, 256, 4096, "resident"), (400, 12, 640, 15424, "resident"),
                                               (1300, 30, 640, 1472, "resident"), (1300, 30, 640, 1344, "tiled")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tokens_of_a_tile_in_lds(avg, E, Kd, N, family, dtype):
    from oracle import oracle as orc
    from vllm_ascend_amd import kernels as K
    from vllm_ascend_amd._lib import W_ENK, load

    R = avg * E
    print(f"tokens in LDS R={R} E={E} K={Kd} N={N} {family} {dtype}", flush=True)
    assert load().moe355_gmm_kernel_name(2, R, Kd, N, E).decode() == f"gmm_{family}_kernel"
    counts = [0, 1, 63, 64, 65, 127, 128, 129] if E > 8 else []
    counts += [160, 161, 192, 193, 256, 257] if E > 24 else []  # the heights of the weight-streaming tiles
    rest = R - sum(counts)
    counts += [rest // (E - len(counts))] * (E - len(counts) - 1)
    counts += [R - sum(counts)]
    counts = torch.tensor(counts)
    cum = counts.cumsum(0)
    g = torch.Generator(device="cuda").manual_seed(R)
    x = torch.randint(-128, 128, (R, Kd), generator=g, dtype=torch.int8, device="cuda")
    w = torch.randint(-128, 128, (E, N, Kd), generator=g, dtype=torch.int8, device="cuda")
    sw = torch.rand(E, N, generator=g, device="cuda") * 0.009 + 0.001
    sx = torch.rand(R, generator=g, device="cuda") * 0.05 + 0.001
    wnz = K.format_cast_nz(w, W_ENK)
    acc = exact_products(x, w, counts)
    assert torch.equal(K.gmm_i32(x, wnz, cum.to("cuda"), 0, N, Kd), acc)
    got = K.gmm2_dequant(x, wnz, sw, sx, cum.to("cuda"), 0, N, Kd, out_dtype=dtype)
    at = torch.repeat_interleave(torch.arange(E), counts).to("cuda")
    want = ((acc.float() * sx[:, None]) * sw[at]).to(dtype)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    if family != "wide":
        return
    # the gate_up product of the same line: the first, a middle and the last rows of every expert against the oracle
    assert load().moe355_gmm_kernel_name(1, R, Kd, N, E) == b"gmm_wide_kernel"
    q, qs = K.gmm1_swiglu_quant(x, wnz, sw, sx, cum.to("cuda"), 0, N, Kd)
    rows = [sorted({int(c) - int(m), int(c) - int(m) // 2 - 1, int(c) - 1}) for c, m in zip(cum, counts) if m]
    picked = torch.tensor(sum(rows, []))
    ends = np.searchsorted(picked.numpy(), cum.numpy())
    q_want, s_want = orc.swiglu_quant(orc.dequant_acc(acc[picked.to("cuda")].cpu().numpy(), sx.cpu()[picked].numpy(),
                                                      sw.cpu().numpy(), ends))
    assert np.array_equal(q.cpu()[picked].numpy(), q_want)
    assert np.array_equal(qs.cpu()[picked].numpy().view(np.uint32), s_want.view(np.uint32))


# ... whose rows end in front of the buffer's, the last ones inside a tile: what lies around the output stays as it is.  Experts of
# one row, whose tile is 128 rows of the next ones
@pytest.mark.parametrize("K_, N", [(256, 2048), (768, 1408)])
@pytest.mark.parametrize("kind", [0, 1])
def test_nothing_is_written_around_the_rows(K_, N, kind):
    from vllm_ascend_amd import kernels as K
    from vllm_ascend_amd._lib import W_ENK, load

    lib, E, R = load(), 16, 38400
    print(f"around the rows K={K_} N={N} kind={kind}", flush=True)
    assert lib.moe355_gmm_kernel_name(2, R, K_, N, E) == b"gmm_resident_kernel"
    counts = torch.tensor([1, 2900, 0, 129, 1, 1, 65, 3000, 128, 1, 4000, 6000, 64, 7000, 13400, 1001])
    rows = int(counts.sum())
    assert rows < R - 600 and rows % 128
    g = torch.Generator(device="cuda").manual_seed(R)
    x = torch.randint(-128, 128, (R, K_), generator=g, dtype=torch.int8, device="cuda")
    w = torch.randint(-128, 128, (E, N, K_), generator=g, dtype=torch.int8, device="cuda")
    sw = torch.rand(E, N, generator=g, device="cuda") * 0.009 + 0.001
    sx = torch.rand(R, generator=g, device="cuda") * 0.05 + 0.001
    wnz = K.format_cast_nz(w, W_ENK)
    gl = (counts if kind else counts.cumsum(0)).to("cuda")
    around = torch.full((R + 512, N), 0x1234, dtype=torch.int16, device="cuda")
    ws = torch.empty(lib.moe355_gmm2_dequant_workspace(R, N, K_, E), dtype=torch.uint8, device="cuda")
    p = lambda t: t.data_ptr()  # noqa: E731
    assert lib.moe355_gmm2_dequant(p(x), p(wnz), p(sw), p(sx), p(gl), kind, R, K_, N, E, p(around[256]), K._dt(x.bfloat16(), "out"),
                                   p(ws), ws.numel(), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert bool((around[:256] == 0x1234).all()) and bool((around[256 + rows:] == 0x1234).all())
    at = torch.repeat_interleave(torch.arange(E), counts).to("cuda")
    want = ((exact_products(x, w, counts).float() * sx[:rows, None]) * sw[at]).to(torch.bfloat16)
    assert torch.equal(around[256:256 + rows], want.view(torch.int16))


# Weight-streaming tiles for a product of 14 MiB per expert and 896 columns of them, up to 256 rows per expert: tall tiles
@pytest.mark.parametrize("avg,E,N,family", [(144, 63, 7168, "wide"), (145, 63, 7168, "tiled"), (145, 64, 7168, "wide"),
                                            (256, 64, 7168, "wide"), (257, 64, 7168, "tiled"), (145, 80, 7104, "tiled")])
def test_rows_of_weight_streaming_tiles(avg, E, N, family):
    test_tokens_of_a_tile_in_lds(avg, E, 2048, N, family, torch.bfloat16)


# and of several tall tiles per expert, where an expert's weights are several times an XCD's L2
@pytest.mark.parametrize("avg,E,Kd,N,family", [(257, 16, 4096, 8192, "wide"), (511, 19, 2048, 7168, "tiled"),
                                               (512, 19, 2048, 7168, "wide"), (700, 19, 2048, 7232, "wide"),
                                               (384, 96, 5120, 4096, "wide")])
def test_several_weight_streaming_tiles_of_an_expert(avg, E, Kd, N, family):
    test_tokens_of_a_tile_in_lds(avg, E, Kd, N, family, torch.bfloat16)


# and where they begin when there are columns for several rounds of the chip
@pytest.mark.parametrize("avg,E,Kd,N,family", [(39, 512, 4096, 576, "tiled"), (40, 512, 4096, 576, "wide"), (40, 511, 4096, 576, "tiled"),
                                               (16, 1024, 7168, 576, "tiled"), (17, 1024, 7168, 576, "wide"),
                                               (16, 1024, 5120, 576, "tiled"), (17, 1024, 5120, 576, "wide"),
                                               (27, 228, 4096, 4160, "tiled"), (28, 228, 4096, 4160, "wide"),
                                               (71, 128, 2048, 7168, "tiled"), (72, 128, 2048, 7168, "wide"),
                                               (39, 179, 3072, 5184, "tiled"), (40, 179, 3072, 5184, "wide")])
def test_few_rows_on_weight_streaming_tiles(avg, E, Kd, N, family):
    test_tokens_of_a_tile_in_lds(avg, E, Kd, N, family, torch.bfloat16)


# Tall tiles of the weight-streaming family (193 to 256 rows), whose two halves of columns are entries of their own as long as
# the list has room: all of them, some of them; an even and an odd number of column blocks (the second half of the last column
# does not exist); beside tiles of every other height
@pytest.mark.parametrize("Kd,N", [(4096, 192), (4096, 448)])
@pytest.mark.parametrize("counts", [[193] * 8, [256, 193, 255, 194, 200, 220, 193, 256], [512, 0, 3, 509, 40, 0], [700, 192, 161, 129, 1, 0, 64, 33]],
                         ids=["no room", "some room", "room", "all heights"])
def test_halves_of_tall_tiles(counts, Kd, N):
    _check_tall_tiles(counts, Kd, N)


# ... which are those of experts with several tiles; tall ones that are their expert's only tile have one entry.  The number of
# entries of the list (the first word of the workspace), with no room for halves, some, enough
@pytest.mark.parametrize("counts,entries", [([200] * 8, 8), ([256, 193, 255, 194, 200, 220, 193, 256], 8), ([449, 1, 1, 1], 5),
                                            ([449, 500, 40, 0], 7), ([449] * 4 + [1] * 4, 15), ([512, 0, 3, 509, 40, 0], 10),
                                            ([240] * 23 + [257], 25), ([240] * 22 + [257, 0], 45)])
def test_entries_of_tall_tiles(counts, entries):
    from vllm_ascend_amd import kernels as K
    from vllm_ascend_amd._lib import load

    lib, E, R, Kd, N = load(), len(counts), sum(counts), 4096, 192
    print(f"entries of {counts}", flush=True)
    assert lib.moe355_gmm_kernel_name(2, R, Kd, N, E).decode() == "gmm_wide_kernel"
    x = torch.zeros(R, Kd, dtype=torch.int8, device="cuda")
    w = torch.zeros(E, N * Kd, dtype=torch.int8, device="cuda")
    sw, sx = torch.ones(E, N, device="cuda"), torch.ones(R, device="cuda")
    gl = torch.tensor(counts, dtype=torch.int64, device="cuda")
    out = torch.empty(R, N, dtype=torch.bfloat16, device="cuda")
    ws = torch.zeros(lib.moe355_gmm2_dequant_workspace(R, N, Kd, E), dtype=torch.uint8, device="cuda")
    p = lambda t: t.data_ptr()  # noqa: E731
    assert lib.moe355_gmm2_dequant(p(x), p(w), p(sw), p(sx), p(gl), 1, R, Kd, N, E, p(out), K._dt(out, "out"), p(ws), ws.numel(),
                                   torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert int(ws[:4].view(torch.int32)) == entries
    _check_tall_tiles(counts, Kd, N)


# ... and every tile is listed once, the two halves of a tall one next to each other in the same eight entries (workgroup i runs on
# XCD i % 8, and the halves of the gate_up product wait for each other): with and without room for all halves, an even and an odd
# number of whole tall tiles and of others
@pytest.mark.parametrize("experts,mean,skew", [(64, 80, 0.8), (64, 100, 1.1), (65, 120, 1.1), (63, 200, 0.8), (48, 150, 0.3), (64, 64, 0.0),
                                               (33, 250, 0.1), (256, 128, 1.1), (255, 96, 0.8), (6, 240, 0.5), (8, 200, 1.1)])
def test_list_of_tiles_by_length(experts, mean, skew):
    from vllm_ascend_amd import kernels as K
    from vllm_ascend_amd._lib import load

    lib, Kd, N = load(), 4096, 64
    w = torch.zeros(experts, N * Kd, dtype=torch.int8, device="cuda")
    sw = torch.ones(experts, N, device="cuda")
    p = lambda t: t.data_ptr()  # noqa: E731
    seen = set()
    for seed in range(12):
        rng = np.random.default_rng(seed)
        R = experts * mean + seed
        popular = (1.0 + rng.permutation(experts)) ** -skew
        counts = rng.multinomial(R, popular / popular.sum())
        assert lib.moe355_gmm_kernel_name(2, R, Kd, N, experts).decode() == "gmm_wide_kernel"
        x = torch.zeros(R, Kd, dtype=torch.int8, device="cuda")
        sx = torch.ones(R, device="cuda")
        gl = torch.from_numpy(counts.astype(np.int64)).cuda()
        out = torch.empty(R, N, dtype=torch.bfloat16, device="cuda")
        ws = torch.zeros(lib.moe355_gmm2_dequant_workspace(R, N, Kd, experts), dtype=torch.uint8, device="cuda")
        assert lib.moe355_gmm2_dequant(p(x), p(w), p(sw), p(sx), p(gl), 1, R, Kd, N, experts, p(out), K._dt(out, "out"), p(ws), ws.numel(),
                                       torch.cuda.current_stream().cuda_stream) == 0
        words = ws.cpu().numpy()[:ws.numel() // 4 * 4].view(np.int32)
        most = R // 256 + experts
        n, pitch = int(words[0]), -(-most // 64) * 64
        assert n <= most
        listed, begin, end = (words[64 + i * pitch:64 + i * pitch + n].astype(np.int64) for i in range(3))
        expert, first, second = listed & ((1 << 28) - 1), (listed >> 29) & 1, (listed >> 28) & 1
        starts = np.cumsum(counts) - counts
        assert np.array_equal(end, starts[expert] + counts[expert])
        want = {(e, int(starts[e]) + r) for e in range(experts) for r in range(0, int(counts[e]), 256)}
        once = [(int(e), int(b)) for e, b, s in zip(expert, begin, second) if not s]
        assert len(once) == len(want) and set(once) == want
        at = np.flatnonzero(second)
        assert np.array_equal(at - 1, np.flatnonzero(first)) and np.all(at % 2 == 1)
        assert np.array_equal(expert[at], expert[at - 1]) and np.array_equal(begin[at], begin[at - 1])
        tall = sum(int(counts[e]) - (b - int(starts[e])) > 192 for e, b in want)
        seen.add((len(at) == tall, (tall - len(at)) % 2, (len(want) - tall) % 2))
        assert np.all(end[at] - begin[at] > 192)
    print(f"{experts} experts, all in halves / odd whole ones / odd others: {sorted(seen)}", flush=True)


def _check_tall_tiles(counts, Kd, N):
    from oracle import oracle as orc
    from vllm_ascend_amd import kernels as K
    from vllm_ascend_amd._lib import W_ENK, load

    E, R = len(counts), sum(counts)
    print(f"tall tiles {counts} K={Kd} N={N}", flush=True)
    assert load().moe355_gmm_kernel_name(2, R, Kd, N, E).decode() == "gmm_wide_kernel"
    g = torch.Generator().manual_seed(R + N)
    cum = torch.cumsum(torch.tensor(counts, dtype=torch.int64), 0)
    x = torch.randint(-128, 128, (R, Kd), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (E, N, Kd), generator=g, dtype=torch.int8)
    sw = torch.rand(E, N, generator=g) * 0.009 + 0.001
    sx = torch.rand(R, generator=g) * 0.05 + 0.001
    wnz = K.format_cast_nz(w.to("cuda"), W_ENK)
    ref = orc.gmm_i32(x.numpy(), w.numpy(), cum.numpy())
    got = K.gmm2_dequant(x.to("cuda"), wnz, sw.to("cuda"), sx.to("cuda"), cum.to("cuda"), 0, N, Kd)
    q, s = K.gmm1_swiglu_quant(x.to("cuda"), wnz, sw.to("cuda"), sx.to("cuda"), cum.to("cuda"), 0, N, Kd)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().contiguous().view(torch.int16).numpy().view(np.uint16), orc.gmm2_dequant(ref, sx.numpy(), sw.numpy(), cum.numpy()))
    q_want, s_want = orc.swiglu_quant(orc.dequant_acc(ref, sx.numpy(), sw.numpy(), cum.numpy()))
    assert np.array_equal(q.cpu().numpy(), q_want)
    assert np.array_equal(s.cpu().numpy().view(np.uint32), s_want.view(np.uint32))
