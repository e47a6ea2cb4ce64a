"""The grouped GEMMs on both sides of the lines between streaming and the tiles: 1023 / 1024 rows for a small product,
fewer rows than experts / one row per expert for one of more than a GiB, 63 / 64 rows per expert at a long K."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

LINES = [(1023, 128, 256, 128, "stream"), (1024, 128, 256, 128, "tiled"), (1100, 1200, 64, 64, "stream"),
         (63 * 8 + 7, 8, 4096, 128, "tiled"), (64 * 8, 8, 4096, 128, "wide"),
         (287, 288, 2048, 2048, "stream"), (288, 288, 2048, 2048, "tiled")]


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
