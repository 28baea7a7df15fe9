"""The batched personalised sweep where no row stands out (nwgraph_amd/csrc/ppr.hip): rows of up to 256
in-edges are light, longer ones are cut, and a row that does stand out moves the line to 32.  A light row
adds its terms one after the other, all >= 0: 256 additions and 4 roundings of the update a sweep."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = 0.85
SWEEPS = 6
RTOL = SWEEPS * 260 * 2.0**-24


@pytest.mark.parametrize("longest", [256, 257, 300, 64 + 8 * 40, 64 + 8 * 40 + 60])
@pytest.mark.parametrize("n,tile,k,relabel", [(4001, 8, 5, 0), (4001, 16, 18, 1), (4001, 32, 33, 0), (4001, 64, 64, 0),
                                              (135001, 64, 64, 1)])
def test_rows_of_even_length(ctx, n, tile, k, relabel, longest):
    rng = np.random.default_rng(n + longest)
    indeg = rng.integers(30, 51, n)
    special = [0, 1, 7, 8, 9, 16, 17, 31, 32, 33, 64, 65, 127, 128, 129, 255, longest] * 3
    indeg[rng.permutation(n)[: len(special)]] = special
    ptr = np.zeros(n + 1, np.int64)
    ptr[1:] = np.cumsum(indeg)
    col = rng.integers(0, n, ptr[-1])
    deg = np.bincount(col, minlength=n)
    g = ctx.graph_from_csc(ptr.astype(np.uint32), col.astype(np.uint32), deg.astype(np.uint32))
    plan = g.get_plan()
    plan.update(ppr_tile=tile, relabel=relabel, binned=0)
    g.set_plan(**plan)
    seeds = [np.sort(rng.choice(n, 1 + j % 9, replace=False)).astype(np.uint32) for j in range(k)]
    x, its, _ = g.ppr(seeds, D, 0.0, SWEEPS)
    assert np.all(its == SWEEPS)
    row = np.repeat(np.arange(n), indeg)
    for j in sorted({0, k // 2, k - 1}):
        base = np.zeros(n)
        base[seeds[j]] = (1 - D) / len(seeds[j])
        want = np.full(n, 1.0 / n)
        for _ in range(SWEEPS):
            want = base + D * np.bincount(row, weights=want[col] / deg[col], minlength=n)
        assert np.all(np.abs(x[:, j] - want) <= RTOL * want)
    g.close()
