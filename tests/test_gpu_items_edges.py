"""The item sweeps (nwgraph_amd/csrc/items.hip) on inputs that the one-workgroup solves otherwise take, and rows
at the edges of an item's 1020 units: resident solves with kernel timing, which small.hip does not serve,
the allocation-free call above its 4096 rows, and a union with one graph too large for a workgroup, whose
items then hold rows of more graphs than the 64 whose L1 changes meet in LDS.  Bounds as in
test_gpu_items.py."""
import numpy as np
import pytest

from kernel_names import kernels
from test_gpu_items import D, SWEEPS, _csc, _fp64, _noalloc

pytestmark = pytest.mark.gpu

KINDS = {
    "one vertex": [5],
    "two vertices": [0, 1],
    "no edges": [0] * 700,
    "one long row": [0] * 40 + [1020 * 9 + 1] + [0] * 40,
    "rows of a span": [1020, 1019, 1021, 0, 2040, 2039, 2041, 0, 0, 10200, 3, 1018] * 4,
    "a span of rows": [1] * 510 + [0] * 1020 + [2] * 340 + [1] * 509,
    "spans of empty rows": ([0] * 1019 + [1022] + [0] * 17 + [5000]) * 3,
}


@pytest.mark.parametrize("relabel", [0, 1])
@pytest.mark.parametrize("kind", list(KINDS))
def test_resident(ctx, kind, relabel):
    n, ptr, col, deg = _csc(KINDS[kind], 5)
    want, err = _fp64(n, ptr, col, deg, D, SWEEPS)
    g = ctx.graph_from_csc(ptr, col, deg)
    g.set_plan(binned=0, relabel=relabel)
    got, info = g.pagerank(D, 0.0, SWEEPS, kernel_timing=True)
    bound = 3 * 2.0**-24 / (1 - D) * want.sum()
    assert info["iterations"] == SWEEPS
    assert np.abs(got - want).sum() <= bound
    assert np.abs(info["error_trace"] - np.array(err)).max() <= 2 * bound
    assert kernels(lambda: g.pagerank(D, 0.0, SWEEPS, kernel_timing=True))["pr_item_kernel"] == SWEEPS
    g.close()


@pytest.mark.parametrize("front", [0, 1, 4100])
@pytest.mark.parametrize("kind", list(KINDS))
def test_noalloc(ctx, kind, front):
    """4100 rows without in-edges around the kind's, so that items serve the call; `front` of them before it."""
    n, ptr, col, deg = _csc([0] * front + KINDS[kind] + [0] * (4100 - front), 6)
    want, err = _fp64(n, ptr, col, deg, D, SWEEPS)
    got, trace = _noalloc(ctx, n, ptr, col, deg, D, SWEEPS)
    bound = 3 * 2.0**-24 / (1 - D) * want.sum()
    assert np.abs(got - want).sum() <= bound
    assert np.abs(trace - np.array(err)).max() <= 2 * bound
    assert kernels(lambda: _noalloc(ctx, n, ptr, col, deg, D, SWEEPS))["pr_item_kernel"] == SWEEPS


@pytest.mark.parametrize("tiny", [63, 64, 65, 300])
def test_union_of_tiny_graphs_and_a_large_one(ctx, tiny):
    rng = np.random.default_rng(tiny)
    sizes = [[int(d) for d in rng.integers(0, 3, n)] for n in rng.integers(1, 5, tiny)]
    sizes.insert(tiny // 2, [25000, 3] + [1] * 300)
    parts = [_csc(d, 11 + q) for q, d in enumerate(sizes)]
    graphs = [ctx.graph_from_csc(ptr, col, deg) for _, ptr, col, deg in parts]
    mg = ctx.multigraph(graphs)
    stopped = 0
    for thr, sweeps in ((0.0, SWEEPS), (1e-4, 60), (1e-4, 60), (1e-4, 60)):
        got, its, _, _ = mg.pagerank(D, thr, sweeps)
        for q, (n, ptr, col, deg) in enumerate(parts):
            want, err = _fp64(n, ptr, col, deg, D, sweeps)
            bound = 3 * 2.0**-24 / (1 - D) * max(want.sum(), 1.0 / n)
            # stops that float64 sweeps decide: no change as close to the threshold as both errors
            stop = next((k + 1 for k, e in enumerate(err) if e < thr), sweeps)
            if thr and any(abs(e - thr) <= 2 * bound for e in err[:stop]):
                continue
            assert its[q] == (stop if thr else sweeps) or err[int(its[q]) - 1] == 0.0, (q, its[q], stop)
            stopped += int(its[q]) < sweeps
            want = _fp64(n, ptr, col, deg, D, int(its[q]))[0]
            assert np.abs(got[mg.offsets[q] : mg.offsets[q + 1]] - want).sum() <= bound, q
    assert stopped > tiny
    assert kernels(lambda: mg.pagerank(D, 0.0, SWEEPS))["pr_item_many_kernel"] == SWEEPS
    mg.close()
    for g in graphs:
        g.close()
