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
