"""The default plan's choice between the item and the binned sweep between 2 M and 6.3 M edges, which looks
at the degrees: whichever runs, both are exact row sums of the same sweeps, so the scores are the
same bits, and the plan says nothing else than it did."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,per_row,hub", [(210001, 10, 0), (230001, 10, 0), (500001, 8, 0), (500001, 5, 0),
                                           (300001, 12, 40000)])
def test_default_sweep_by_degrees(ctx, n, per_row, hub):
    rng = np.random.default_rng(n + hub)
    m = n * per_row
    src, dst = rng.integers(0, n, m).astype(np.uint32), rng.integers(0, n, m).astype(np.uint32)
    src[:hub] = 7
    g = ctx.graph_from_edges(n, src, dst)
    got, info = g.pagerank(0.85, 1e-4, 20)
    assert g.get_plan()["binned"] == 1 and g.get_plan()["bin_bits"] == 0 and g.get_plan()["relabel"] == (hub > 0)
    for plan in ({"binned": 0}, {"binned": 1, "bin_bits": 13}):
        g.set_plan(**plan)
        want, winfo = g.pagerank(0.85, 1e-4, 20)
        assert winfo["iterations"] == info["iterations"] and np.array_equal(got, want)
    g.close()


@pytest.mark.parametrize("binned", [0, 1])
def test_union_of_skewed_and_plain_graphs(ctx, binned):
    """A union of 2 M edges is swept with its skewed graphs in degree order and the others as they are: every
    graph's scores and stopping sweep are those of its own solve, for a damping beyond the exact sums'
    range (the older kernel) within float sums of the same sweeps."""
    rng = np.random.default_rng(5)
    graphs = []
    for n, per_row, hub in ((60001, 12, 30000), (1, 1, 0), (40000, 9, 0), (3, 2, 0), (90001, 8, 50000), (513, 20, 900)):
        m = n * per_row
        src, dst = rng.integers(0, n, m).astype(np.uint32), rng.integers(0, n, m).astype(np.uint32)
        src[:hub] = n // 3
        graphs.append(ctx.graph_from_edges(n, src, dst))
    mg = ctx.multigraph(graphs)
    assert mg.nnz >= 1 << 20
    mg.set_plan(binned)
    for _ in range(2):
        got, its, _, _ = mg.pagerank(0.85, 1e-4, 30)
        for q, g in enumerate(graphs):
            g.set_plan(binned=0)
            want, info = g.pagerank(0.85, 1e-4, 30)
            assert its[q] == info["iterations"]
            assert np.array_equal(got[mg.offsets[q] : mg.offsets[q + 1]], want), q
    if not binned:
        got, its, _, _ = mg.pagerank(1.01, 0.0, 10)
        for q, g in enumerate(graphs):
            want, _ = g.pagerank(1.01, 0.0, 10)
            # float sums of up to 50,000 terms, tree or serial per row, so each sweep within 4100 * 2^-24 of the sum
            # of its terms, and those of a sweep sum to at most 1.01 |x|_1; errors grow by 1.01 a sweep
            total = np.abs(want).sum(dtype=np.float64)
            err = np.abs(got[mg.offsets[q] : mg.offsets[q + 1]].astype(np.float64) - want).sum()
            assert err <= 2 * 10 * 4100 * 2.0**-24 * 1.01**10 * total, q
    for g in graphs:
        g.close()
