"""The pull form of the weighted solve (wsweep_kernel in nwgraph_amd/csrc/wpr.hip), which serves what the
exact sweeps' bound does not cover: sources whose raw weights sum to 0, negative and un-normalised
weights, teleports and gradients that are not finite.

Bounds: with u = 2^-24 a float row sum of at most M terms is within (M + 1) u of the sum of their absolute
values, products included, and weight normalisation, the update and the base add 5 u of the row's value, so
the error of a sweep's iterate obeys e' <= d |W| e + (M + 6) u (|b| + d |W| |y|), which _solve evaluates
along with the float64 sweeps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = float(np.float32(0.85))
U = 2.0**-24


def _graph(ctx, n, m, seed):
    rng = np.random.default_rng(seed)
    src, dst = rng.integers(0, n, m).astype(np.uint32), rng.integers(0, n, m).astype(np.uint32)
    g = ctx.graph_from_edges(n, src, dst, clean=False)
    ptr, col, _ = g.csc()
    return g, np.repeat(np.arange(n), np.diff(ptr.astype(np.int64))), col, rng


def _normalised(n, col, w):
    with np.errstate(all="ignore"):
        return w.astype(np.float64) / np.bincount(col, weights=w.astype(np.float64), minlength=n)[col]


def _solve(n, to, frm, wn, b, y, sweeps):
    """float64 sweeps y <- b + d sum w y over the edges frm -> to, and their error bound"""
    terms = max(np.bincount(to, minlength=n).max(), np.bincount(frm, minlength=n).max())
    e = np.zeros(n)
    with np.errstate(all="ignore"):
        for _ in range(sweeps):
            ay = np.abs(b) + D * np.bincount(to, weights=np.abs(wn * y[frm]), minlength=n)
            e = D * np.bincount(to, weights=np.abs(wn) * e[frm], minlength=n) + (terms + 6) * U * ay
            y = b + D * np.bincount(to, weights=wn * y[frm], minlength=n)
    return y, e


def _same(got, want, bound):
    """values within the bound where they are finite, the same NaN and infinities elsewhere"""
    fin = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
    assert np.all(np.abs(got[fin] - want[fin]) <= np.broadcast_to(bound, want.shape)[fin])


def _raw_gradient(n, row, col, w, wn, lam, x):
    s = np.bincount(col, weights=w.astype(np.float64), minlength=n)
    with np.errstate(all="ignore"):
        t = x * np.bincount(col, weights=D * lam[row] * wn, minlength=n)
        return (D * lam[row] * x[col] - t[col]) / s[col]


SIZES = [(300, 2000), (5003, 30000)]  # one workgroup's and the item sweep's sizes


@pytest.mark.parametrize("n,m", SIZES)
def test_source_without_weight_shows_nan(ctx, n, m):
    """A source whose raw weights are all 0 (or sum past the largest float) has normalised weights of 0 / 0:
    scores, adjoint and raw gradients that they reach are NaN, all others are the values of float64 sweeps."""
    g, row, col, rng = _graph(ctx, n, m, n)
    for value in (0.0, 3e38):
        w = rng.uniform(0.1, 1.0, m).astype(np.float32)
        for u in (5, 77):
            assert (col == u).sum() > 1
            w[col == u] = value
        g.set_weights(w)
        wn = _normalised(n, col, w)
        wn[(col == 5) | (col == 77)] = np.nan
        x0 = rng.uniform(0.1, 1.0, n).astype(np.float32) / np.float32(n)
        c = rng.normal(size=n).astype(np.float32)
        for _ in range(3):  # launched one by one, captured, replayed
            x, fi = g.wpr_forward(None, D, 0.0, 2)
            want, e = _solve(n, row, col, wn, np.full(n, (1 - D) / n), np.full(n, 1.0 / n), 2)
            assert fi["iterations"] == 2 and np.isnan(want).any() and np.isfinite(want).any()
            _same(x, want, e)
            gw, gv, bi = g.wpr_backward(x0, c, D, 0.0, 2)
            lam, el = _solve(n, col, row, wn, c.astype(np.float64), c.astype(np.float64), 2)
            assert bi["iterations"] == 2 and np.isnan(lam).any() and np.isfinite(lam).any()
            _same(gv, (1 - D) * lam, el + 2 * U * np.abs(lam))
            ge = _raw_gradient(n, row, col, w, wn, lam, x0.astype(np.float64))
            assert np.array_equal(np.isnan(gw), np.isnan(ge)) and np.isfinite(ge).any()
    g.close()


def test_source_without_weight_in_the_binned_sweep(ctx):
    """A binned plan drops the mass of such a source, as if its edges were not there."""
    n, m = SIZES[1]
    g, row, col, rng = _graph(ctx, n, m, 3)
    g.set_plan(binned=1, bin_bits=13)
    w = rng.uniform(0.1, 1.0, m).astype(np.float32)
    w[col == 5] = 0.0
    g.set_weights(w)
    wn = _normalised(n, col, w)
    wn[col == 5] = 0.0
    x, _ = g.wpr_forward(None, D, 0.0, 12)
    _same(x, *_solve(n, row, col, wn, np.full(n, (1 - D) / n), np.full(n, 1.0 / n), 12))
    g.close()


@pytest.mark.parametrize("n,m", SIZES + [(40001, 300000)])
@pytest.mark.parametrize("kind", ["negative", "as given"])
def test_weights_outside_the_exact_sweeps(ctx, n, m, kind):
    """Negative raw weights and weights that are not normalised: forward and adjoint against float64 sweeps."""
    g, row, col, rng = _graph(ctx, n, m, n + 1)
    g.set_plan(binned=0)
    outdeg = np.bincount(col, minlength=n)
    if kind == "negative":  # about one edge in ten; a source's sum stays away from 0
        w = rng.uniform(0.2, 1.0, m)
        w[rng.random(m) < 0.1] *= -0.02
        first = np.unique(col, return_index=True)[1]
        w[first] = 1.0
    else:
        w = rng.uniform(0.1, 1.5, m) / outdeg[col]
    w = w.astype(np.float32)
    g.set_weights(w, normalize=kind == "negative")
    wn = _normalised(n, col, w) if kind == "negative" else w.astype(np.float64)
    v = rng.random(n)
    v = (v / v.sum()).astype(np.float32)
    c = rng.normal(size=n).astype(np.float32)
    for _ in range(3):
        x, fi = g.wpr_forward(v, D, 0.0, 23)
        want, e = _solve(n, row, col, wn, (1 - D) * v.astype(np.float64), np.full(n, 1.0 / n), 23)
        assert fi["iterations"] == 23
        _same(x, want, e)
        gw, gv, bi = g.wpr_backward(x, c, D, 0.0, 23, raw_weights=False)
        lam, el = _solve(n, col, row, wn, c.astype(np.float64), c.astype(np.float64), 23)
        assert bi["iterations"] == 23
        _same(gv, (1 - D) * lam, el + 2 * U * np.abs(lam))
        x64 = x.astype(np.float64)
        _same(gw, D * lam[row] * x64[col], D * el[row] * np.abs(x64[col]) + 3 * U * np.abs(lam[row] * x64[col]))
    g.close()


@pytest.mark.parametrize("plan", [{}, {"binned": 1, "bin_bits": 13}])
@pytest.mark.parametrize("n,m", SIZES)
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_teleport_or_gradient_not_finite(ctx, n, m, bad, plan):
    """One entry of the teleport or the gradient is not finite: the exact sweep gives way to the pull sweep,
    which shows it where it reaches; solves on the same graph before and after are not touched by it."""
    g, row, col, rng = _graph(ctx, n, m, n + 2)
    if plan:
        g.set_plan(**plan)
    w = rng.uniform(0.1, 1.0, m).astype(np.float32)
    g.set_weights(w)
    wn = _normalised(n, col, w)
    v = (rng.uniform(0.5, 1.5, n) / n).astype(np.float32)
    c = rng.normal(size=n).astype(np.float32)
    x0 = (rng.uniform(0.1, 1.0, n) / n).astype(np.float32)
    vb, cb = v.copy(), c.copy()
    vb[7] = cb[7] = bad
    for vv, cc in ((v, c), (vb, cb), (vb, cb), (vb, cb), (v, c)):
        x, fi = g.wpr_forward(vv, D, 0.0, 3)
        want, e = _solve(n, row, col, wn, (1 - D) * vv.astype(np.float64), np.full(n, 1.0 / n), 3)
        _same(x, want, e)
        gw, gv, bi = g.wpr_backward(x0, cc, D, 0.0, 3)
        lam, el = _solve(n, col, row, wn, cc.astype(np.float64), cc.astype(np.float64), 3)
        _same(gv, (1 - D) * lam, el + 2 * U * np.abs(lam))
        ge = _raw_gradient(n, row, col, w, wn, lam, x0.astype(np.float64))
        assert np.array_equal(np.isnan(gw), np.isnan(ge))
        assert fi["iterations"] == bi["iterations"] == 3
    g.close()
