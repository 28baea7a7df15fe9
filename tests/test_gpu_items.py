"""The item sweep (nwgraph_amd/csrc/items.hip) at the edges of its work items: rows just below,
at and above an item's span, rows over many items, runs of empty rows, item counts of one and
just past the switch between 64 and 256 lanes.  Scores are held to float64 sweeps: row sums are
exact, so a sweep rounds each score three times (x / deg, the row sum, the update) and damps
what it inherits by d, at most 3 * 2^-24 / (1 - d) of the score vector in all."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = 0.85
SWEEPS = 12


def _csc(indeg, seed):
    indeg = np.asarray(indeg, np.int64)
    n = indeg.size
    rng = np.random.default_rng(seed)
    ptr = np.zeros(n + 1, np.int64)
    ptr[1:] = np.cumsum(indeg)
    col = rng.integers(0, n, ptr[-1])
    return n, ptr.astype(np.uint32), col.astype(np.uint32), np.bincount(col, minlength=n).astype(np.uint32)


def _fp64(n, ptr, col, deg, d, sweeps):
    row = np.repeat(np.arange(n), np.diff(ptr.astype(np.int64)))
    x = np.full(n, 1.0 / n)
    err = []
    for _ in range(sweeps):
        z = np.bincount(row, weights=x[col] / deg[col], minlength=n)
        y = (1 - d) / n + d * z
        err.append(np.abs(y - x).sum())
        x = y
    return x, err


def _noalloc(ctx, n, ptr, col, deg, d, sweeps):
    import torch
    from nwgraph_amd import _lib

    dev = [torch.from_numpy(a.astype(np.int32)).cuda() for a in (ptr, col, deg)]
    x = torch.full((n,), -1.0, device="cuda")
    info = _lib.PrInfo()
    err = np.zeros(sweeps)
    info.error_trace = err.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    info.error_trace_len = sweeps
    torch.cuda.synchronize()
    ctx.check(ctx.lib.nwg_pagerank_f32_noalloc(ctx.handle, n, col.size, dev[0].data_ptr(), dev[1].data_ptr(),
                                               dev[2].data_ptr(), x.data_ptr(), d, 0.0, sweeps, ctypes.byref(info)))
    assert int(info.iterations) == sweeps
    return x.cpu().numpy(), err


def _degrees(kind):
    rng = np.random.default_rng(3)
    if kind == "one vertex":
        return [5]
    if kind == "no edges":
        return [0] * 700
    if kind == "one long row":
        return [0] * 40 + [252 * 9 + 1] + [0] * 40
    if kind == "around the span of 64 lanes":
        return [252, 251, 253, 0, 0, 504, 503, 505, 1, 252, 252, 0, 2520, 7] * 8
    if kind == "switch to 256 lanes":  # 2^18 units: the largest graph of 64-lane items
        return [1] * (1 << 17)
    if kind == "around the span of 256 lanes":
        return [1020, 1019, 1021, 0, 2040, 2041, 0, 0, 10200, 3, 1018] * 20 + [2] * (1 << 16)
    if kind == "empty rows between long ones":
        return ([0] * 3000 + [1500] + [0] * 17 + [5000]) * 20 + [1] * 130000
    return np.minimum(rng.zipf(2.0, 90001), 30000)  # skewed


KINDS = ["one vertex", "no edges", "one long row", "around the span of 64 lanes", "switch to 256 lanes",
         "around the span of 256 lanes", "empty rows between long ones", "skewed"]


@pytest.mark.parametrize("kind", KINDS)
def test_noalloc_items_match_float64(ctx, kind):
    n, ptr, col, deg = _csc(_degrees(kind), 5)
    want, err = _fp64(n, ptr, col, deg, D, SWEEPS)
    got, trace = _noalloc(ctx, n, ptr, col, deg, D, SWEEPS)
    bound = 3 * 2.0**-24 / (1 - D) * want.sum()
    assert np.abs(got - want).sum() <= bound
    # each sweep's L1 change is off by at most twice the iterates' distance from float64
    assert np.abs(trace - np.array(err)).max() <= 2 * bound


@pytest.mark.parametrize("relabel", [0, 1])
@pytest.mark.parametrize("kind", KINDS)
def test_resident_items_match_float64(ctx, kind, relabel):
    """The resident solve's pull plan, over two segments of sweeps (20, then 8 at a time)."""
    n, ptr, col, deg = _csc(_degrees(kind), 5)
    sweeps = 23
    want, err = _fp64(n, ptr, col, deg, D, sweeps)
    g = ctx.graph_from_csc(ptr, col, deg)
    g.set_plan(binned=0, relabel=relabel)
    got, info = g.pagerank(D, 0.0, sweeps)
    bound = 3 * 2.0**-24 / (1 - D) * want.sum()
    assert info["iterations"] == sweeps
    assert np.abs(got - want).sum() <= bound
    assert np.abs(info["error_trace"] - np.array(err)).max() <= 2 * bound
    g.close()


@pytest.mark.parametrize("n", [12007, 70001])  # 64- and 256-lane items
def test_resident_items_stop_and_personalise(ctx, n):
    rng = np.random.default_rng(n)
    n, ptr, col, deg = _csc(np.minimum(rng.zipf(2.0, n), 3000), 6)
    v = rng.random(n)
    v = (v / v.sum()).astype(np.float32)
    row = np.repeat(np.arange(n), np.diff(ptr.astype(np.int64)))
    x = np.full(n, 1.0 / n)
    for it in range(1, 60):
        y = (1 - D) * v.astype(np.float64) + D * np.bincount(row, weights=x[col] / deg[col], minlength=n)
        done = np.abs(y - x).sum() < 1e-4
        x = y
        if done:
            break
    g = ctx.graph_from_csc(ptr, col, deg)
    g.set_plan(binned=0)
    for _ in range(2):
        got, info = g.pagerank(D, 1e-4, 100, teleport=v)
        assert info["iterations"] == it
        assert np.abs(got - x).sum() <= 3 * 2.0**-24 / (1 - D) * x.sum()
    g.close()


@pytest.mark.parametrize("kind", ["tiny", "long rows between tiny ones", "one each"])
def test_items_of_many_graphs(ctx, kind):
    """Items over rows of several graphs, of more than the 64 whose L1 changes meet in LDS, and rows over
    several items that end among other graphs' rows: every graph's scores and stopping sweep."""
    rng = np.random.default_rng(7)
    if kind == "tiny":
        sizes = [[int(d) for d in rng.integers(0, 3, n)] for n in list(rng.integers(1, 5, 300)) + [1, 900]]
    elif kind == "long rows between tiny ones":
        sizes = []
        for big in (1019, 1020, 1021, 2040, 5000, 30000):
            sizes += [[1, 2, 0], [big], [0, big, 1, big + 1, 0], [3]]
    else:
        sizes = [[int(d) for d in np.minimum(rng.zipf(1.8, n), 4000)] for n in (300, 1020, 5000, 40001)]
    parts = [_csc(d, 11 + q) for q, d in enumerate(sizes)]
    graphs = [ctx.graph_from_csc(ptr, col, deg) for _, ptr, col, deg in parts]
    mg = ctx.multigraph(graphs)
    for thr, sweeps in ((0.0, SWEEPS), (1e-4, 60), (1e-4, 60)):
        got, its, _, _ = mg.pagerank(D, thr, sweeps)
        for q, (n, ptr, col, deg) in enumerate(parts):
            want, err = _fp64(n, ptr, col, deg, D, sweeps)
            bound = 3 * 2.0**-24 / (1 - D) * max(want.sum(), 1.0 / n)
            # stops that float64 sweeps decide: no change as close to the threshold as both errors
            clear = [abs(e - thr) > 2 * bound for e in err]
            stop = next((k + 1 for k, e in enumerate(err) if e < thr), sweeps)
            if all(clear[:stop]) or thr == 0.0:
                assert its[q] == (stop if thr else sweeps) or err[int(its[q]) - 1] == 0.0, (q, its[q], stop)
                want = _fp64(n, ptr, col, deg, D, int(its[q]))[0]
                assert np.abs(got[mg.offsets[q] : mg.offsets[q + 1]] - want).sum() <= bound, q
    for g in graphs:
        g.close()


def test_weighted_items_with_a_fold_launch(ctx):
    """More than 1024 items: the L1 change is folded by a launch between the sweeps; stops as the change
    of float64 sweeps says, away from the threshold."""
    rng = np.random.default_rng(4)
    n, m = 400001, 900000
    src, dst = rng.integers(0, n, m).astype(np.uint32), rng.integers(0, n, m).astype(np.uint32)
    g = ctx.graph_from_edges(n, src, dst, clean=False)
    ptr, col, _ = g.csc()
    row = np.repeat(np.arange(n), np.diff(ptr.astype(np.int64)))
    w = rng.uniform(0.1, 1.0, m).astype(np.float32)
    wn = w / np.bincount(col, weights=w.astype(np.float64), minlength=n)[col]
    x, err = np.full(n, 1.0 / n), []
    for _ in range(40):
        y = (1 - D) / n + D * np.bincount(row, weights=wn * x[col], minlength=n)
        err.append(np.abs(y - x).sum())
        x = y
    g.set_weights(w)
    for it in (3, 20, 21, 30):  # the geometric mean of two changes: a factor of about 1 / sqrt(d) away
        got, info = g.wpr_forward(None, D, float(np.sqrt(err[it - 1] * err[it - 2])), 40)
        assert info["iterations"] == it
    g.close()


@pytest.mark.parametrize("side", ["in", "out"])  # the degrees are those of the CSC's or the CSR's rows
@pytest.mark.parametrize("kind", KINDS)
def test_weighted_items_match_float64(ctx, kind, side):
    """Weighted forward and adjoint over items, and the raw-weight gradient over the CSR's items.  With
    u = 2^-24: a forward sweep rounds each (positive) score six times at most, weight normalisation
    included, so 12 of them stay within 72 u of every score; an adjoint sweep is off by at most 6 u of
    the largest |lambda|, damped by d; the gradient's two terms are at most d |lambda| x_u / s_u."""
    deg = np.asarray(_degrees(kind), np.int64)
    n, m = deg.size, int(deg.sum())
    rng = np.random.default_rng(8)
    a, b = np.repeat(np.arange(n), deg), rng.integers(0, n, m)
    src, dst = (b, a) if side == "in" else (a, b)
    g = ctx.graph_from_edges(n, src.astype(np.uint32), dst.astype(np.uint32), clean=False)
    ptr, col, _ = g.csc()
    row = np.repeat(np.arange(n), np.diff(ptr.astype(np.int64)))
    w = rng.uniform(0.1, 1.0, m).astype(np.float32)
    c = rng.normal(size=n).astype(np.float32)
    g.set_weights(w)
    x, fi = g.wpr_forward(None, D, 0.0, SWEEPS)
    gw, gv, bi = g.wpr_backward(x, c, D, 0.0, SWEEPS)
    assert fi["iterations"] == bi["iterations"] == SWEEPS
    u = 2.0**-24
    total = np.bincount(col, weights=w.astype(np.float64), minlength=n)
    wn = w / total[col]
    want = np.full(n, 1.0 / n)
    ferr = []
    for _ in range(SWEEPS):
        y = (1 - D) / n + D * np.bincount(row, weights=wn * want[col], minlength=n)
        ferr.append(np.abs(y - want).sum())
        want = y
    assert np.all(np.abs(x - want) <= 72 * u * want)
    assert np.abs(fi["error_trace"] - np.array(ferr)).max() <= 2 * 72 * u * max(want.sum(), 1.0)
    lam, lmax = c.astype(np.float64), np.abs(c).max()
    for _ in range(SWEEPS):
        lam = c + D * np.bincount(col, weights=wn * lam[row], minlength=n)
        lmax = max(lmax, np.abs(lam).max())
    assert np.abs(gv - (1 - D) * lam).max() <= (6 / (1 - D) + 2) * u * lmax
    t = want * np.bincount(col, weights=D * lam[row] * wn, minlength=n)
    ge = (D * lam[row] * want[col] - t[col]) / total[col] if m else np.zeros(0)
    assert np.all(np.abs(gw - ge) <= 2 * (72 + 6 / (1 - D) + 8) * u * D * lmax * (want / np.maximum(total, 0.1))[col])
    g.close()


def test_noalloc_damping_above_one_keeps_float_sums(ctx):
    """The exact sums cover damping factors in [0, 1]; above, the float row sums serve the call.  A
    sweep is off by at most m * 2^-24 for a row of m float terms and 3 * 2^-24 for its other
    roundings, and multiplies what it inherits by at most d."""
    d = 1.01
    n, ptr, col, deg = _csc(_degrees("around the span of 64 lanes"), 5)
    want, _ = _fp64(n, ptr, col, deg, d, SWEEPS)
    got, _ = _noalloc(ctx, n, ptr, col, deg, d, SWEEPS)
    assert np.abs(got - want).sum() <= SWEEPS * d**SWEEPS * (2520 + 3) * 2.0**-24 * np.abs(want).sum()
