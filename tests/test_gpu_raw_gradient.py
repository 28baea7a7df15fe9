"""The gradient with respect to raw weights where it is exactly 0: a source with one out-edge sends it all its
mass whatever the weight (also one whose reciprocal is past the largest float), and so does one whose
edges lead to vertices of equal lambda."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = 0.85


@pytest.mark.parametrize("n,plan", [(400, {}), (6000, {}), (6000, {"binned": 1, "bin_bits": 13}), (70001, {})])
def test_only_out_edge_has_no_gradient(ctx, n, plan):
    rng = np.random.default_rng(n)
    one = np.arange(0, n, 2)
    src = np.concatenate([one, np.repeat(np.arange(1, n, 2), 6)]).astype(np.uint32)
    dst = rng.integers(0, n, src.size).astype(np.uint32)
    g = ctx.graph_from_edges(n, src, dst, clean=False)
    if plan:
        g.set_plan(**plan)
    ptr, col, _ = g.csc()
    row = np.repeat(np.arange(n), np.diff(ptr.astype(np.int64)))
    w = rng.uniform(0.1, 1.0, col.size).astype(np.float32)
    w[np.isin(col, one[::5])] = 1e-42
    g.set_weights(w)
    x, _ = g.wpr_forward(None, D, 0.0, 15)
    c = rng.normal(size=n).astype(np.float32)
    gw, gv, _ = g.wpr_backward(x, c, D, 0.0, 15)
    single = col % 2 == 0
    assert np.all(gw[single] == 0.0)
    # the others against float64, given the solve's own lambda: four roundings of either term and one of
    # their difference
    u = 2.0**-24
    wn = w / np.bincount(col, weights=w.astype(np.float64), minlength=n)[col]
    lam = gv.astype(np.float64) / (1 - D)  # two more
    s = np.bincount(col, weights=w.astype(np.float64), minlength=n)
    dl = D * lam[row]
    mean = np.bincount(col, weights=dl * wn, minlength=n)[col]
    size = np.bincount(col, weights=np.abs(dl) * wn, minlength=n)[col] + np.abs(dl)
    a = x.astype(np.float64)[col] / s[col]
    assert np.all(np.abs(gw - a * (dl - mean))[~single] <= (8 * u * size * a)[~single])
    g.close()


@pytest.mark.parametrize("raw", [True, False])
@pytest.mark.parametrize("n", [400, 6000])
def test_teleport_gradient_over_the_scores(ctx, n, raw):
    """grad_teleport may be written where the scores were, over one segment of sweeps and over several, and
    when the solve starts again with another sweep (a gradient of one vertex that is not finite)."""
    import torch

    rng = np.random.default_rng(n)
    src, dst = rng.integers(0, n, 6 * n).astype(np.uint32), rng.integers(0, n, 6 * n).astype(np.uint32)
    g = ctx.graph_from_edges(n, src, dst)
    g.set_weights(rng.uniform(0.1, 1.0, g.nnz).astype(np.float32))
    x0, _ = g.wpr_forward(None, D, 0.0, 15)
    for sweeps, bad in ((10, False), (45, False), (10, True)):
        c = rng.normal(size=n).astype(np.float32)
        if bad:
            c[3] = np.inf
        want_w, want_v, _ = g.wpr_backward(x0, c, D, 0.0, sweeps, raw_weights=raw)
        x, cd = torch.from_numpy(x0).cuda(), torch.from_numpy(c).cuda()
        gw = torch.zeros(g.nnz, device="cuda")
        torch.cuda.synchronize()
        g.wpr_backward_device(x.data_ptr(), cd.data_ptr(), gw.data_ptr(), x.data_ptr(), D, 0.0, sweeps,
                              raw_weights=raw)
        assert np.array_equal(gw.cpu().numpy(), want_w, equal_nan=True)
        assert np.array_equal(x.cpu().numpy(), want_v, equal_nan=True)
    g.close()
