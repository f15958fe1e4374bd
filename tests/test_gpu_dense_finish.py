"""Segments with more ks than one radix select answers are sorted in LDS in
registers (4 to 32 keys a thread), or by the global radix sort above that: sizes
around each step, every rank and a few ranks."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _bits(a):
    return a.view(np.uint64 if a.dtype.itemsize == 8 else np.uint32)


# whole inputs small enough to be one segment
@pytest.mark.parametrize("dtype", ["float32", "float64", "uint32", "int32"])
@pytest.mark.parametrize("n", [9, 63, 64, 65, 255, 256, 257, 1000, 4095, 4096, 4097, 8192, 8193, 16384, 16385, 32768])
def test_one_segment(dtype, n, gpu_ctx):
    import ggms
    for dist, p0 in (("uniform", 0.0), ("mod_index", 5.0)):
        x = ggms.generate(dtype, dist, n, 3, p0)
        h = x.cpu().numpy()
        for nk in (8, 9, min(n, 1000), n):
            ks = (np.arange(nk, dtype=np.int64) * 7 % n + 1).astype(np.uint32)
            got = gpu_ctx.select(x, ks, "iterative")
            assert np.array_equal(_bits(got), _bits(oracle.sort_and_choose(h, ks, threads=8))), (dist, nk)


# few buckets: dense segments of about n / buckets keys, up to past the sort's capacity
@pytest.mark.parametrize("dtype,buckets", [(d, b) for d in ("float32", "float64") for b in (16, 40, 200, 2000)])
@pytest.mark.parametrize("schedule", [0, 1])
def test_dense_segments_of_a_pass(dtype, buckets, schedule, gpu_ctx):
    import ggms
    n = 400_003
    x = ggms.generate(dtype, "normal", n, 9)
    ks = ggms.generate_ks("even", 3000, n, 1)
    o = ggms.default_opts(num_buckets=buckets, schedule=schedule)
    for alg in ("bucket", "iterative"):
        got = gpu_ctx.select(x, ks, alg, o)
        assert np.array_equal(_bits(got), _bits(oracle.sort_and_choose(x.cpu().numpy(), ks, threads=8)))
