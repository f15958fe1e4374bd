"""Mixtures of components narrow beside their distance from zero put many ranges
into one cell of the first pass's table, a few components or more than it has
tables for: exact results with every splitter and both first-pass layouts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(a):
    return a.view(np.uint64 if a.dtype.itemsize == 8 else np.uint32)


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("components,sigma", [(3, 1e-3), (8, 1e-2), (50, 1e-4)])
@pytest.mark.parametrize("splitter", [0, 1, 2])
def test_exact(dtype, components, sigma, splitter, gpu_ctx):
    import ggms
    import torch
    n = 1_000_003
    rng = np.random.default_rng(components)
    mu = rng.uniform(-100, 100, components)
    h = (mu[rng.integers(0, components, n)] + sigma * rng.standard_normal(n)).astype(dtype)
    x = torch.from_numpy(h).cuda()
    order = np.sort(h)
    for nk in (301, 8192):
        ks = ggms.generate_ks("even", nk, n, 1)
        want = order[n - ks.astype(np.int64)]
        for alg in ("iterative", "bucket"):
            got = gpu_ctx.select(x, ks, alg, ggms.default_opts(splitter=splitter, learned_pieces=128 if splitter else 0,
                                                               num_pivots=0 if splitter else 129))
            assert np.array_equal(_bits(got), _bits(want)), (alg, nk)


@pytest.mark.parametrize("dtype,pivots", [("float32", 940), ("float32", 985), ("uint32", 1024), ("float64", 500)])
@pytest.mark.parametrize("nk", [1, 301, 8192, 9000])
def test_largest_tables(dtype, pivots, nk, gpu_ctx):
    """the most buckets and many pivots fit every kernel's LDS"""
    import ggms
    n = 2_000_003
    x = ggms.generate(dtype, "uniform" if dtype == "uint32" else "normal", n, 5)
    order = np.sort(x.cpu().numpy())
    ks = ggms.generate_ks("even", nk, n, 1)
    want = order[n - ks.astype(np.int64)]
    for first_pass in (0, 1, 2):
        for schedule in (0, 1):
            o = ggms.default_opts(num_buckets=16384, num_pivots=pivots, sample_size=16384, first_pass=first_pass,
                                  schedule=schedule)
            for alg in ("iterative", "bucket"):
                got = gpu_ctx.select(x, ks, alg, o)
                assert np.array_equal(_bits(got), _bits(want)), (first_pass, schedule, alg)
