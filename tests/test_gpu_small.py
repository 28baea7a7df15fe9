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
@pytest.mark.parametrize("n,m", [(1, 3), (2, 4096), (1023, 4095), (1024, 4096), (1025, 4096), (1024, 4097), (4096, 8191),
                                 (3001, 8192), (3001, 8193), (4096, 16384), (4097, 16384), (4095, 16385)])
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
