"""The linear splitter cuts pieces whose sample crowds in part of their key span
into more ranges: results stay exact over sample sizes, pivot counts (below, at
and above the range that is cut) and distributions, infinities included."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _bits(a):
    return a.view(np.uint64 if a.dtype.itemsize == 8 else np.uint32)


def _data(dtype, dist, n):
    rng = np.random.default_rng(11)
    x = rng.standard_normal(n)
    if dist == "half":
        x = np.abs(x)
    elif dist == "two_scales":  # half the keys in a millionth of the rest's span
        x[::2] *= 1e-6
    elif dist == "steps":  # long runs of one value inside a piece
        x = np.floor(x * 4) + (rng.random(n) < 0.3) * rng.random(n) * 1e-3
    elif dist == "nonfinite":
        x[:5] = [np.inf, -np.inf, np.inf, -np.inf, 0.0]
    return x.astype(dtype)


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("dist", ["normal", "half", "two_scales", "steps", "nonfinite"])
def test_exact(dtype, dist, gpu_ctx):
    import ggms
    import torch
    n = 300_007
    h = _data(dtype, dist, n)
    x = torch.from_numpy(h).cuda()
    ks = ggms.generate_ks("even", 301, n, 1)
    want = oracle.sort_and_choose(h, ks, threads=8)
    for sample, pivots in ((0, 0), (64, 4), (512, 17), (1024, 3), (1024, 5), (2048, 64), (4096, 65), (2048, 200)):
        for buckets in (0, 64, 2000):
            for schedule in (0, 1):
                o = ggms.default_opts(sample_size=sample, num_pivots=pivots, num_buckets=buckets, schedule=schedule)
                got = gpu_ctx.select(x, ks, "iterative", o)
                assert np.array_equal(_bits(got), _bits(want)), (sample, pivots, buckets, schedule)
