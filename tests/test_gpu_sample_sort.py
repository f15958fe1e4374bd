"""The first-pass sample's in-register sort, seen through the range table: with
many pivots the range starts are order statistics of the sample, which is
redrawn here from Philox and sorted with numpy."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _keys(v):
    b = 8 * v.dtype.itemsize
    u = v.view(np.uint64 if b == 64 else np.uint32)
    one = u.dtype.type(1)
    return np.where(u >> u.dtype.type(b - 1) != 0, ~u, u | (one << u.dtype.type(b - 1)))


# four keys a thread in one to sixteen waves, then eight and sixteen keys a
# thread; the last size only with 4-byte keys
@pytest.mark.parametrize("dtype,sample", [(d, s) for d in ("float32", "float64")
                                          for s in (200, 256, 257, 512, 1000, 1024, 2048, 4096, 5000, 8192, 16384)
                                          if d == "float32" or s <= 8192])
def test_range_starts_are_sample_order_statistics(dtype, sample, gpu_ctx):
    import ggms
    n, seed, P = 3_000_001, 77 + sample, min(1000 if dtype == "float32" else 400, sample // 2)
    x = ggms.generate(dtype, "normal", n, 5)
    o = ggms.default_opts(num_pivots=P, sample_size=sample, seed=seed)
    ranges, _ = gpu_ctx.first_pass(x, o)
    key = [(seed & 0xFFFFFFFF) ^ 0x67676D73, seed >> 32]
    draw = np.array([oracle.philox([i, 0, 2, 0], key)[0] for i in range(sample)], dtype=np.uint64)
    s = np.sort(_keys(x.cpu().numpy()[(draw * np.uint64(n)) >> np.uint64(32)]))
    eo = max(1, (22 * sample + 512) // 1024)
    po = (sample - 2 * eo) // (P - 3)
    idx = [0, eo - 1] + [min(po * (i - 1) + eo - 1, sample - 1) for i in range(2, P - 2)] + [sample - eo - 1, sample - 1]
    q = np.unique(s[idx])
    starts = ranges["lo"].astype(q.dtype)
    assert np.all(starts[1:] > starts[:-1])
    assert np.all(np.isin(q, starts))
    # between the sample's extremes, beside the pivots: the key after a pivot value that repeats
    extra = starts[~np.isin(starts, q) & (starts > q[0]) & (starts < q[-1])]
    assert np.all(np.isin(extra, q + q.dtype.type(1)))
