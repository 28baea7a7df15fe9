"""Whole solves in one workgroup (nwgraph_amd/csrc/small.hip): row and edge counts just below, at and above
those of its variants, rows over many lanes and waves, solves over several launches, many graphs at
once.  Scores are held to float64 sweeps as in test_gpu_items.py: row sums are exact, so a sweep
rounds each score three times, at most 3 * 2^-24 / (1 - d) of the score vector in all."""
import numpy as np
import pytest

from test_gpu_items import D, _csc, _fp64, _noalloc

pytestmark = pytest.mark.gpu

BOUND = 3 * 2.0**-24 / (1 - D)


def _degrees(n, m, kind):
    """n in-degrees that sum to m"""
    rng = np.random.default_rng(n + m)
    if kind == "one row":
        d = np.zeros(n, np.int64)
        d[n // 2] = m
    elif kind == "few long rows":  # with empty ones between
        d = np.zeros(n, np.int64)
        at = rng.choice(n, min(n, 7), replace=False)
        d[at] = m // at.size
        d[at[0]] += m - d.sum()
    else:
        d = np.bincount(np.minimum(rng.integers(0, n, m), rng.integers(0, n, m)), minlength=n)
    return d


@pytest.mark.parametrize("kind", ["skewed", "one row", "few long rows"])
@pytest.mark.parametrize("n,m", [(1, 3), (2, 4096), (1023, 4095), (1024, 4096), (1025, 4096), (1024, 4097),
                                 (4096, 8191), (3001, 8192), (3001, 8193), (4096, 16384), (4097, 16384),
                                 (4095, 16385), (4096, 20480), (4096, 20481)])
def test_scores_and_changes(ctx, n, m, kind):
    n, ptr, col, deg = _csc(_degrees(n, m, kind), n)
    sweeps = 12
    want, err = _fp64(n, ptr, col, deg, D, sweeps)
    bound = BOUND * max(want.sum(), 1.0 / n)
    g = ctx.graph_from_csc(ptr, col, deg)
    for relabel in (0, 1):
        g.set_plan(binned=0, relabel=relabel)
        got, info = g.pagerank(D, 0.0, sweeps)
        assert np.abs(got - want).sum() <= bound and info["iterations"] == sweeps
        assert np.abs(info["error_trace"] - np.array(err)).max() <= 2 * bound
    got, trace = _noalloc(ctx, n, ptr, col, deg, D, sweeps)
    assert np.abs(got - want).sum() <= bound
    assert np.abs(trace - np.array(err)).max() <= 2 * bound
    g.close()


def test_stops_personalises_and_goes_on_over_launches(ctx):
    from nwgraph_amd import NwgError

    n, ptr, col, deg = _csc(_degrees(2000, 9000, "skewed"), 2)
    row = np.repeat(np.arange(n), np.diff(ptr.astype(np.int64)))
    v = np.random.default_rng(1).random(n)
    v = (v / v.sum()).astype(np.float32)
    x, errs = np.full(n, 1.0 / n), []
    for _ in range(60):
        y = (1 - D) * v.astype(np.float64) + D * np.bincount(row, weights=x[col] / deg[col], minlength=n)
        errs.append(np.abs(y - x).sum())
        x = y
        if errs[-1] < 1e-4:
            break
    g = ctx.graph_from_csc(ptr, col, deg)
    for relabel in (0, 1):
        g.set_plan(binned=0, relabel=relabel)
        got, info = g.pagerank(D, 1e-4, 100, teleport=v)
        assert info["iterations"] == len(errs) and np.abs(got - x).sum() <= BOUND
        with pytest.raises(NwgError):
            g.pagerank(D, 1e-4, 100, teleport=np.full(n, 1.01 / n, np.float32))
    # 2500 sweeps are three launches; the scores have long settled
    settled = _fp64(n, ptr, col, deg, D, 200)[0]
    got, info = g.pagerank(D, 0.0, 2500)
    assert info["iterations"] == 2500 and np.abs(got - settled).sum() <= BOUND * max(settled.sum(), 1.0)
    got, trace = _noalloc(ctx, n, ptr, col, deg, D, 2500)
    assert np.abs(got - settled).sum() <= BOUND * max(settled.sum(), 1.0)
    g.close()


def test_many_graphs_one_workgroup_each(ctx):
    shapes = [(1, 0), (1, 5), (300, 2000), (1024, 24576), (4096, 20000), (77, 24000), (4, 0)]
    parts = [_csc(_degrees(n, m, k), n) for n, m in shapes for k in ("skewed", "few long rows")]
    graphs = [ctx.graph_from_csc(ptr, col, deg) for _, ptr, col, deg in parts]
    mg = ctx.multigraph(graphs)
    for thr in (0.0, 1e-4):
        for _ in range(2):
            got, its, _, _ = mg.pagerank(D, thr, 40)
            for q, (n, ptr, col, deg) in enumerate(parts):
                want, err = _fp64(n, ptr, col, deg, D, 40)
                bound = BOUND * max(want.sum(), 1.0 / n)
                stop = next((k + 1 for k, e in enumerate(err) if e < thr), 40)
                if thr == 0.0 or all(abs(e - thr) > 2 * bound for e in err[:stop]):
                    # without a threshold a change of exactly 0 never stops a solve either
                    assert its[q] == stop, (q, its[q], stop)
                    want = _fp64(n, ptr, col, deg, D, stop)[0]
                    assert np.abs(got[mg.offsets[q] : mg.offsets[q + 1]] - want).sum() <= bound, q
    for g in graphs:
        g.close()


@pytest.mark.parametrize("kind", ["skewed", "one row", "few long rows"])
@pytest.mark.parametrize("n,m", [(1, 3), (1024, 4096), (1025, 4096), (1024, 4097), (4096, 8192), (3001, 8193),
                                 (4096, 16384), (4097, 16384), (4095, 16385), (4096, 20480), (4096, 20481)])
def test_weighted_solves(ctx, n, m, kind):
    """Forward and adjoint with the bounds of test_weighted_items_match_float64 (u = 2^-24: 72 u of every
    score after 12 sweeps; the adjoint off by 6 u of the largest |lambda|, damped by d), stops away
    from the threshold, and a solve over two launches, whose scores have settled to 6 u / (1 - d) of
    every score."""
    sweeps, u = 12, 2.0**-24
    rng = np.random.default_rng(m)
    src, dst = rng.integers(0, n, m), np.repeat(np.arange(n), _degrees(n, m, kind))
    g = ctx.graph_from_edges(n, src.astype(np.uint32), dst.astype(np.uint32), clean=False)
    ptr, col, _ = g.csc()
    row = np.repeat(np.arange(n), np.diff(ptr.astype(np.int64)))
    w = rng.uniform(0.1, 1.0, m).astype(np.float32)
    wn = w / np.bincount(col, weights=w.astype(np.float64), minlength=n)[col]
    v = rng.random(n).astype(np.float32)
    g.set_weights(w)

    def iterate(b, x, at, to, count):
        err = []
        for _ in range(count):
            y = b + D * np.bincount(to, weights=wn * x[at], minlength=n)
            err.append(np.abs(y - x).sum())
            x = y
        return x, err

    want, err = iterate((1 - D) * v.astype(np.float64), np.full(n, 1.0 / n), col, row, sweeps)
    x, fi = g.wpr_forward(v, D, 0.0, sweeps)
    assert np.all(np.abs(x - want) <= 72 * u * want) and fi["iterations"] == sweeps
    c = rng.normal(size=n).astype(np.float32)
    gw, gv, bi = g.wpr_backward(x, c, D, 0.0, sweeps)
    lam, lmax = c.astype(np.float64), np.abs(c).max()
    for _ in range(sweeps):
        lam = c + D * np.bincount(col, weights=wn * lam[row], minlength=n)
        lmax = max(lmax, np.abs(lam).max())
    assert np.abs(gv - (1 - D) * lam).max() <= (6 / (1 - D) + 2) * u * lmax
    for it in (2, 5, 9):
        if err[it - 1] > 1e-4 * np.abs(want).sum() and err[it - 1] < 0.95 * err[it - 2]:
            _, info = g.wpr_forward(v, D, float(np.sqrt(err[it - 1] * err[it - 2])), 40)
            assert info["iterations"] == it
            thr = float(np.sqrt(err[it - 1] * err[it - 2])) / np.abs(v.astype(np.float64)).sum()
            _, info = g.wpr_forward(v, D, thr, 40, relative=True)
            assert info["iterations"] == it
    settled, _ = iterate((1 - D) * v.astype(np.float64), want, col, row, 200)
    x, info = g.wpr_forward(v, D, 0.0, 1500)
    assert info["iterations"] == 1500 and np.all(np.abs(x - settled) <= 6 / (1 - D) * u * settled)
    g.close()


@pytest.mark.parametrize("what", ["id", "decreasing", "end", "out-degree"])
def test_noalloc_refuses_what_its_check_finds(ctx, what):
    """The solve is queued behind the check and leaves the scores alone when it fails."""
    import torch
    from nwgraph_amd import NwgError, _lib

    n, ptr, col, deg = _csc(_degrees(1000, 5000, "skewed"), 3)
    if what == "id":
        col[777] = n
    elif what == "decreasing":
        ptr[500], ptr[501] = ptr[501] + 1, ptr[500]
    elif what == "end":
        ptr[n] -= 1
    else:
        deg[col[0]] -= 1
    dev = [torch.from_numpy(a.astype(np.int32)).cuda() for a in (ptr, col, deg)]
    x = torch.full((n,), -1.0, device="cuda")
    torch.cuda.synchronize()
    for given in (True, False):
        if what == "out-degree" and not given:
            continue
        with pytest.raises(NwgError) as e:
            ctx.check(ctx.lib.nwg_pagerank_f32_noalloc(ctx.handle, n, col.size, dev[0].data_ptr(), dev[1].data_ptr(),
                                                       dev[2].data_ptr() if given else None, x.data_ptr(), D, 0.0, 20,
                                                       None))
        assert e.value.code == _lib.NWG_EINVAL
        assert torch.all(x == -1.0)
