"""The splitter network's tiled kernels at the edges of their tiles (64 samples
a workgroup, up to 256 workgroups, partial sums in a workspace of 65 floats a
sample) against float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MI, MH = 65, 32
MP = MH * MI + 2 * MH + 1


# 66 and 67: the first size whose workspace holds two partials; 16384 and
# 16385: one tile a workgroup, then a workgroup with two
@pytest.mark.parametrize("nb", [1, 15, 16, 63, 64, 65, 66, 67, 127, 129, 1000, 16384, 16385, 40007])
def test_tiles_match_float64(nb, gpu_ctx):
    import ctypes as C
    import torch
    import ggms
    lib = ggms._lib.load()
    P = lambda t: C.c_void_p(t.data_ptr())
    rng = np.random.default_rng(nb)
    w = (rng.standard_normal(MP) * 0.2).astype(np.float32)
    x = rng.random((nb, MI)).astype(np.float32)
    y = rng.random(nb).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).cuda()
    wd, xd, yd = dev(w), dev(x), dev(y)
    # exactly the documented workspace, with guard words behind it and the results
    words = int(lib.ggms_mlp_workspace_floats(nb))
    out = torch.full((nb + 64,), 7.0, device="cuda")
    g = torch.full((MP + 64,), 7.0, device="cuda")
    loss = torch.full((65,), 7.0, device="cuda")
    work = torch.full((words + 64,), 7.0, device="cuda")
    assert lib.ggms_mlp_forward(P(wd), P(xd), nb, P(out), None) == 0
    assert lib.ggms_mlp_loss_grad(P(wd), P(xd), P(yd), nb, P(g), P(loss), P(work), None) == 0
    for t, n in ((out, nb), (g, MP), (loss, 1), (work, words)):
        assert bool((t[n:] == 7.0).all())

    W = w.astype(np.float64)
    W1, b1, W2, b2 = W[:MH * MI].reshape(MH, MI), W[MH * MI:MH * MI + MH], W[MH * MI + MH:-1], W[-1]
    X, Y = x.astype(np.float64), y.astype(np.float64)
    z = X @ W1.T + b1
    a = np.maximum(z, 0)
    p = 1 / (1 + np.exp(-(a @ W2 + b2)))
    d = (p - Y) * p * (1 - p) / nb
    on = np.where(z > 0, 1.0, 0.0)
    dz = d[:, None] * W2 * on
    ref = np.concatenate([(dz.T @ X).ravel(), dz.sum(0), a.T @ d, [d.sum()]])
    # fp32 sums of at most 68 products and then of at most ~100 partials, and the
    # rounding of the terms: 1e-5 of the sum of their sizes; a unit within 1e-5 of
    # zero may be taken as on or off (its whole term)
    near = np.abs(z) < 1e-5
    size = np.abs(d)[:, None] * np.abs(W2)
    tol = 1e-5 * np.concatenate([((size * on).T @ X).ravel(), (size * on).sum(0), a.T @ np.abs(d), [np.abs(d).sum()]])
    tol += np.concatenate([((size * near).T @ X).ravel(), (size * near).sum(0), np.zeros(MH + 1)]) + 1e-12
    # the error of p shows in (p - y) p (1 - p) / nb of every sample
    tol += 2e-6 * np.concatenate([(np.abs(W2) * on).T @ X, ((np.abs(W2) * on).sum(0))[:, None], a.sum(0)[:, None]],
                                 axis=1).ravel().max() / nb
    got = g[:MP].cpu().numpy().astype(np.float64)
    assert np.all(np.abs(got - ref) <= tol), np.max(np.abs(got - ref) / tol)
    assert np.max(np.abs(out[:nb].cpu().numpy() - p)) <= 2e-6
    l = np.mean(0.5 * (p - Y) ** 2)
    assert abs(float(loss[0]) - l) <= 1e-5 * l + 1e-9
    # the same inputs give the same bits: no sum depends on the order of atomics
    g2 = torch.empty(MP, device="cuda")
    assert lib.ggms_mlp_loss_grad(P(wd), P(xd), P(yd), nb, P(g2), P(loss), P(work), None) == 0
    assert bool((g2 == g[:MP]).all())
