"""The binned weighted sweep where the item sweep would serve the graph: plans that name a bin size.  New weights
reach the solves' recorded loops (launched, recorded and replayed for every set of weights, so that a
loop recorded over the old layout would be replayed), and forward, adjoint and gradients hold to float64.
Each test looks at the names of the kernels that ran."""
import numpy as np
import pytest

from kernel_names import kernels

pytestmark = pytest.mark.gpu

D = float(np.float32(0.85))
U = 2.0**-24


def _seen(call, name):
    return any(k.startswith(name) for k in kernels(call))


def _float64(n, to, frm, wn, b, y, sweeps):
    for _ in range(sweeps):
        y = b + D * np.bincount(to, weights=wn * y[frm], minlength=n)
    return y


@pytest.mark.parametrize("bits", [13, 14])
def test_new_weights_reach_the_recorded_binned_solves(ctx, bits):
    """Per sweep at most 3 * 2^-24 of rounding (weight, product, row update) is added to the score vector and
    2^-24 per weight to its normalisation; what a sweep inherits is damped by d.  The adjoint's products have
    both signs: its vector is off by as much of the largest |lambda|."""
    g = ctx.rmat(15, 16, seed=3)
    g.set_plan(binned=1, bin_bits=bits)
    ptr, col, _ = g.csc()
    n, row = g.n, np.repeat(np.arange(g.n), np.diff(ptr.astype(np.int64)))
    rng = np.random.default_rng(1)
    c = rng.normal(size=n).astype(np.float32)
    sweeps, other = 12, None
    for step in range(4):
        w = rng.uniform(0.1, 1.0, g.nnz).astype(np.float32)
        g.set_weights(w)
        other = ctx.rmat(13 + step % 2, 16, seed=step)  # shifts what the next layout is allocated from
        wn = w / np.bincount(col, weights=w.astype(np.float64), minlength=n)[col]
        want = _float64(n, row, col, wn, np.full(n, (1 - D) / n), np.full(n, 1.0 / n), sweeps)
        lam = _float64(n, col, row, wn, c.astype(np.float64), c.astype(np.float64), sweeps)
        for _ in range(3):
            x, info = g.wpr_forward(None, D, 0.0, sweeps)
            assert info["iterations"] == sweeps
            assert np.abs(x - want).sum() <= 6 * U / (1 - D) * want.sum()
            _, gv, _ = g.wpr_backward(x, c, D, 0.0, sweeps)
            assert np.abs(gv - (1 - D) * lam).max() <= (6 / (1 - D) + 2) * U * np.abs(lam).max()
    assert _seen(lambda: g.wpr_forward(None, D, 0.0, sweeps), f"pr_bin_kernel<false,0,true,{bits}>")
    other.close()
    g.close()


@pytest.mark.parametrize("scale,plan,name", [(12, dict(binned=1, bin_bits=13), "pr_bin_kernel<false,0,true,13>"),
                                             (12, dict(binned=1, bin_bits=14), "pr_bin_kernel<false,0,true,14>"),
                                             (12, dict(binned=0), "wpr_item_kernel"),
                                             (18, dict(binned=1, bin_bits=13), "pr_bin_kernel<false,0,true,13>"),
                                             (18, dict(binned=0), "wsweep_kernel")])
def test_weighted_sweeps_against_float64(ctx, scale, plan, name):
    """Every form of the weighted solve on R-MAT graphs of 53 K and 3.9 M edges: the forward from a teleport, the
    adjoint of gradients of both signs at two scales, edge and raw-weight gradients.  The pull sweep's float
    sums take up to 10^4 terms, in a tree of lanes of 256 at least: within (10^4 / 256 + 16) 2^-24 a sweep."""
    g = ctx.rmat(scale, 16, seed=8)
    g.set_plan(**plan)
    ptr, col, _ = g.csc()
    n, row = g.n, np.repeat(np.arange(g.n), np.diff(ptr.astype(np.int64)))
    rng = np.random.default_rng(scale)
    w = rng.uniform(0.1, 1.0, g.nnz).astype(np.float32)
    g.set_weights(w)
    s = np.bincount(col, weights=w.astype(np.float64), minlength=n)
    wn = w / s[col]
    v = rng.uniform(size=n)
    v = (v / v.sum()).astype(np.float32)
    sweeps = 23
    want = _float64(n, row, col, wn, (1 - D) * v.astype(np.float64), np.full(n, 1.0 / n), sweeps)
    grow = 60 * U / (1 - D)
    for rep in range(3):
        x, info = g.wpr_forward(v, D, 0.0, sweeps)
        assert info["iterations"] == sweeps
        assert np.abs(x - want).sum() <= grow * want.sum()
    for amp in (1.0, 1000.0):
        c = (amp * rng.normal(size=n)).astype(np.float32)
        lam = _float64(n, col, row, wn, c.astype(np.float64), c.astype(np.float64), sweeps)
        lmax = max(np.abs(lam).max(), np.abs(c).max())
        gw, gv, _ = g.wpr_backward(x, c, D, 0.0, sweeps, raw_weights=False)
        assert np.abs(gv - (1 - D) * lam).max() <= (grow + 2 * U) * lmax
        x64 = x.astype(np.float64)[col]
        assert np.all(np.abs(gw - D * lam[row] * x64) <= (grow + 4 * U) * lmax * x64)
        gw, _, _ = g.wpr_backward(x, c, D, 0.0, sweeps)
        mean = np.bincount(col, weights=D * lam[row] * wn, minlength=n)[col]
        assert np.all(np.abs(gw - (D * lam[row] - mean) * x64 / s[col]) <= 2 * (grow + 8 * U) * lmax * x64 / s[col])
    assert _seen(lambda: g.wpr_backward(x, c, D, 0.0, sweeps), name)
    assert _seen(lambda: g.wpr_forward(v, D, 0.0, sweeps), name)
    g.close()
