"""The index maps of the dispatch against numpy's stable sort: at the borders of a chunk (1024 pairs), of the one-launch
form (65536 pairs, 512 experts), with every pair on one expert and with pairs outside the expert range."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("skew", ["uniform", "one expert", "dropped"])
@pytest.mark.parametrize("tokens, k, experts", [(1, 1, 1), (1023, 1, 8), (1024, 1, 256), (205, 5, 128), (8192, 8, 128),
                                                (65536, 1, 3), (4099, 8, 512), (8193, 8, 128), (700, 2, 513)])
def test_maps_equal_a_stable_sort(tokens, k, experts, skew):
    from vllm_ascend_amd import kernels as K

    rng = np.random.default_rng(tokens + experts)
    ids = rng.integers(0, experts, (tokens, k)).astype(np.int32)
    if skew == "one expert":
        ids[:] = experts - 1
    elif skew == "dropped":
        ids[rng.random((tokens, k)) < 0.3] = experts
        ids[rng.random((tokens, k)) < 0.1] = -1
    flat = ids.reshape(-1)
    kept = (flat >= 0) & (flat < experts)
    order = np.flatnonzero(kept)[np.argsort(flat[kept], kind="stable")]
    want_dst = np.full(flat.size, flat.size, dtype=np.int32)
    want_dst[order] = np.arange(order.size)
    counts = np.bincount(flat[kept], minlength=experts)
    for kind in (0, 1):
        dst, row_token, num = K.route_map(torch.from_numpy(ids).to(DEV), experts, kind)
        assert np.array_equal(dst.cpu().numpy(), want_dst)
        assert np.array_equal(row_token.cpu().numpy()[: order.size], order // k)
        assert np.array_equal(num.cpu().numpy(), counts if kind == 1 else np.cumsum(counts))


# from 20480 pairs on, four ids per load: one pair less, remainders of one to three, the last one alone in its 4096; 16 and 8
# counters per expert (256 / 257 experts, one)
@pytest.mark.parametrize("skew", ["uniform", "one expert", "dropped"])
@pytest.mark.parametrize("tokens, k, experts", [(20479, 1, 256), (20480, 1, 256), (20481, 1, 257), (4097, 5, 1), (10241, 2, 512),
                                                (32767, 1, 64), (32769, 1, 64), (65535, 1, 128)])
def test_maps_of_many_pairs(tokens, k, experts, skew):
    test_maps_equal_a_stable_sort(tokens, k, experts, skew)
