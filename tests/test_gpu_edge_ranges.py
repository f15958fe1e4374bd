"""Keys beyond the sample's extremes: the edge ranges give small integers a
bucket each, so a value the sample missed costs no further pass."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _check(ctx, x, ks, alg, opts):
    got = ctx.select(x, ks, alg, opts)
    want = oracle.sort_and_choose(x.cpu().numpy(), ks, threads=8)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    return ctx.stats()


@pytest.mark.parametrize("dtype", ["uint32", "int32"])
def test_missed_small_integers_take_one_pass(dtype, gpu_ctx):
    import ggms
    import torch
    # 2048 values: a sample of 1024 misses both of its extreme values in most draws
    v = torch.arange(1 << 20, device="cuda", dtype=torch.int64) * 7919 % 2048
    x = (v if dtype == "uint32" else v - 1000).to(torch.int32)
    x = x.view(torch.uint32) if dtype == "uint32" else x
    ks = ggms.generate_ks("even", 4096, 1 << 20, 1)
    for seed in range(6):
        st = _check(gpu_ctx, x, ks, "iterative", ggms.default_opts(seed=seed, first_pass=2))
        assert st["passes"] == 1 and st["n_kept"] == [0]


# sample sizes and bucket counts at which the edge ranges are smallest (one
# bucket each) and the sample's outer span is one key or a few
@pytest.mark.parametrize("buckets,sample,pivots", [(16, 8, 3), (16, 64, 17), (100, 65, 17), (14336, 1024, 17), (16384, 16384, 17)])
@pytest.mark.parametrize("dist", ["uniform", "cauchy", "mod_index", "constant"])
def test_extreme_ranks(buckets, sample, pivots, dist, gpu_ctx):
    import ggms
    n = 300_007
    x = ggms.generate("float32", dist, n, 11, 3.0)
    ks = np.concatenate([np.arange(1, 40), np.arange(n - 40, n + 1), [n // 2]]).astype(np.uint32)
    for alg in ("iterative", "bucket", "distributed"):
        _check(gpu_ctx, x, ks, alg, ggms.default_opts(num_buckets=buckets, sample_size=sample, num_pivots=pivots))
