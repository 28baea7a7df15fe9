"""New weights on a resident graph of the binned weighted sweep's size: the captured solve loops must
follow the new weighted layout, wherever its arrays are allocated."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = 0.85


def _fp64_forward(n, ptr, col, w, sweeps):
    row = np.repeat(np.arange(n), np.diff(ptr.astype(np.int64)))
    wn = w / np.bincount(col, weights=w, minlength=n)[col]
    x = np.full(n, 1.0 / n)
    for _ in range(sweeps):
        x = (1 - D) / n + D * np.bincount(row, weights=wn * x[col], minlength=n)
    return x


def test_new_weights_reach_the_captured_solves(ctx):
    """Per sweep at most 3 * 2^-24 of rounding (weight, product, row update) is added to the score
    vector and 2^-24 per weight to its normalisation; what a sweep inherits is damped by d."""
    g = ctx.rmat(15, 16, seed=3)
    assert g.nnz >= 1 << 18
    ptr, col, _ = g.csc()
    rng = np.random.default_rng(1)
    sweeps, other = 12, None
    for step in range(4):
        w = rng.uniform(0.1, 1.0, g.nnz).astype(np.float32)
        g.set_weights(w)
        other = ctx.rmat(13 + step % 2, 16, seed=step)  # shifts what the next layout is allocated from
        x, info = g.wpr_forward(None, D, 0.0, sweeps)
        want = _fp64_forward(g.n, ptr, col, w.astype(np.float64), sweeps)
        assert info["iterations"] == sweeps
        assert np.abs(x - want).sum() <= 6 * 2.0**-24 / (1 - D) * want.sum()
    other.close()
    g.close()
