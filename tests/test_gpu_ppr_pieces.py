"""The batched personalised sweep (nwgraph_amd/csrc/ppr.hip) at the edges of its work split: rows just
below, at and above the cut between light and heavy ones, a piece, a row split by source slice and a
workgroup of pieces; vectors that fill no group of four; one and four rows per lane group; score
arrays at no 16-byte boundary.  Every term is >= 0, so a score's relative error grows by at most the
roundings of one sweep: no sum takes more than 32 additions in a piece, 128 pieces in a workgroup and
40 partials, and the update 4 roundings, 204 * 2^-24 a sweep."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = 0.85
SWEEPS = 6
RTOL = SWEEPS * 204 * 2.0**-24
DEGREES = [0, 1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 34, 63, 64, 65, 95, 127, 129, 255, 256, 257, 511, 1023, 1025, 5000,
           20000]


def _case(n, seed):
    rng = np.random.default_rng(seed)
    indeg = rng.integers(0, 4, n)
    indeg[rng.permutation(n)[: 4 * len(DEGREES)]] = DEGREES * 4
    ptr = np.zeros(n + 1, np.int64)
    ptr[1:] = np.cumsum(indeg)
    col = rng.integers(0, n, ptr[-1])
    return ptr.astype(np.uint32), col.astype(np.uint32), np.bincount(col, minlength=n).astype(np.uint32)


def _fp64(n, ptr, col, deg, ids):
    row = np.repeat(np.arange(n), np.diff(ptr.astype(np.int64)))
    base = np.zeros(n)
    base[ids] = (1 - D) / len(ids)
    x = np.full(n, 1.0 / n)
    for _ in range(SWEEPS):
        x = base + D * np.bincount(row, weights=x[col] / deg[col], minlength=n)
    return x


@pytest.mark.parametrize("n,tile,k,relabel", [(6001, 8, 1, 0), (6001, 8, 21, 1), (6001, 16, 18, 0), (6001, 32, 35, 1),
                                              (6001, 64, 64, 0), (6001, 64, 131, 1), (6001, 16, 301, 0), (540001, 64, 64, 0),
                                              (540001, 32, 63, 1)])
def test_rows_at_the_edges_of_the_split(ctx, n, tile, k, relabel):
    import torch

    ptr, col, deg = _case(n, seed=n + tile)
    g = ctx.graph_from_csc(ptr, col, deg)
    plan = g.get_plan()
    plan.update(ppr_tile=tile, relabel=relabel)
    g.set_plan(**plan)
    rng = np.random.default_rng(k)
    seeds = [np.sort(rng.choice(n, 1 + j % 9, replace=False)).astype(np.uint32) for j in range(k)]
    buf = torch.full((n * k + 1,), -1.0, device="cuda")
    torch.cuda.synchronize()
    g.ppr_device(seeds, buf.data_ptr(), D, 0.0, SWEEPS)
    x = buf[: n * k].view(n, k).cpu().numpy()
    for j in sorted({0, k // 2, k - 1}):
        ref = _fp64(n, ptr, col, deg, seeds[j])
        assert np.all(np.abs(x[:, j] - ref) <= RTOL * ref), (j, np.max(np.abs(x[:, j] - ref) / np.maximum(ref, 1e-30)))
    if n < 10000:  # the same scores, four bytes further on
        g.ppr_device(seeds, buf.data_ptr() + 4, D, 0.0, SWEEPS)
        assert np.array_equal(buf[1:].view(n, k).cpu().numpy(), x)
