"""Inputs of at most the finish capacity take one launch: lengths around the
sort network's sizes and the select's, ranks on the host and on the device, bad
ranks, unaligned bases, graph capture."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _bits(a):
    return a.view(np.uint64 if a.dtype.itemsize == 8 else np.uint32)


@pytest.mark.parametrize("dtype", ["float32", "float64", "uint32", "int32"])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 4096, 4097, 8192, 12345, 16384, 16385, 32767, 32768])
@pytest.mark.parametrize("schedule", [0, 1])
def test_host_and_device_ranks(dtype, n, schedule, gpu_ctx):
    import ggms
    import torch
    buf = ggms.generate(dtype, "cauchy" if dtype.startswith("f") else "uniform", n + 3, n)
    o = ggms.default_opts(schedule=schedule)
    for off in (0, 1, 3):
        x = buf[off:off + n]
        h = x.cpu().numpy()
        for nk in (1, 8, 9, 1500):
            ks = (np.arange(nk, dtype=np.int64) * 977 % n + 1).astype(np.uint32)
            want = _bits(oracle.sort_and_choose(h, ks, threads=8))
            assert np.array_equal(_bits(gpu_ctx.select(x, ks, "bucket", o)), want)
            out = torch.empty(nk, dtype=x.dtype, device="cuda")
            gpu_ctx.select_device(x, torch.from_numpy(ks.view(np.int32)).cuda().view(torch.uint32), out, "iterative", o)
            torch.cuda.synchronize()
            assert np.array_equal(_bits(out.cpu().numpy()), want)


@pytest.mark.parametrize("n,nk", [(1000, 5), (1000, 50), (20000, 5), (20000, 2000), (32768, 8)])
def test_bad_rank_on_the_device_leaves_the_others(n, nk, gpu_ctx):
    import ggms
    import torch
    x = ggms.generate("uint32", "uniform", min(n, 16384), 3)
    n = x.numel()
    ks = (np.arange(nk, dtype=np.int64) * 31 % n + 1).astype(np.uint32)
    bad = [0, nk // 2, nk - 1]
    for j, v in zip(bad, (0, n + 1, 0xFFFFFFFF)):
        ks[j] = v
    out = torch.full((nk,), 12345, dtype=torch.int32, device="cuda").view(torch.uint32)
    d = torch.from_numpy(ks.view(np.int32)).cuda().view(torch.uint32)
    with pytest.raises(ggms.GGMSError) as e:
        gpu_ctx.select_device(x, d, out, "iterative")
    assert e.value.status == ggms.EINVAL
    good = np.setdiff1d(np.arange(nk), bad)
    got = out.cpu().numpy()
    assert np.array_equal(got[good], oracle.sort_and_choose(x.cpu().numpy(), ks[good], threads=8))
    assert np.all(got[bad] == 12345)
    # the next call starts clean
    gpu_ctx.select(x, [1, n], "iterative")


def test_graph_replays(gpu_ctx):
    import ggms
    import torch
    n, nk = 5000, 33
    ctx = ggms.Context(0)
    o = ggms.default_opts(schedule=1)
    assert ctx.lib.ggms_ctx_reserve(ctx.h, 0, n, nk, o) == 0
    x = ggms.generate("float32", "normal", n, 1)
    ks = np.arange(1, nk + 1, dtype=np.uint32) * 100
    d = torch.from_numpy(ks.view(np.int32)).cuda().view(torch.uint32)
    out = torch.empty(nk, device="cuda")
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        o.stream = s.cuda_stream
        ctx.select_device(x, d, out, "iterative", o)
    for seed in range(4):
        x.copy_(ggms.generate("float32", "normal", n, 100 + seed))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), oracle.sort_and_choose(x.cpu().numpy(), ks, threads=8))
        assert ctx.lib.ggms_ctx_device_status(ctx.h) == 0
