"""The automatic bucket count follows the number of ks, the span of their ranks
and the number of keys: every side of its lines gives the exact answers, on both
schedules."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(a):
    return a.view(np.uint64 if a.dtype.itemsize == 8 else np.uint32)


# one-pass: 256 / 257 ks; the root of nk n on each side of its lines
@pytest.mark.parametrize("dtype,n", [("float32", 70_001), ("float32", 3_000_017), ("float64", 1_200_003), ("uint32", 9_000_001)])
@pytest.mark.parametrize("kdist", ["even", "top", "window"])
def test_both_sides(dtype, n, kdist, gpu_ctx):
    import ggms
    x = ggms.generate(dtype, "uniform" if dtype == "uint32" else "normal", n, 5)
    h = x.cpu().numpy()
    order = np.sort(h)
    for nk in (1, 101, 256, 257, 1200, 3583, 3584):
        if kdist == "even":
            ks = ggms.generate_ks("even", nk, n, 1)
        else:
            first = 0 if kdist == "top" else n // 2
            ks = (first + 1 + np.arange(nk)).astype(np.uint32)
        want = order[n - ks.astype(np.int64)]
        for alg in ("iterative", "bucket", "distributed"):
            for schedule in (0, 1):
                got = gpu_ctx.select(x, ks, alg, ggms.default_opts(schedule=schedule))
                assert np.array_equal(_bits(got), _bits(want)), (alg, nk, schedule)
