"""Device memory kept between calls (nwgraph_amd/csrc/devpool.hpp): blocks of released graphs, of a failed
call and of other streams must not show in what later calls compute, and a graph may outlive its
context."""
import threading

import numpy as np
import pytest

import nwgraph_amd
import pyoracle as O
from nwgraph_amd import NwgError

pytestmark = pytest.mark.gpu


def _solve(c, scale, seed):
    g = c.rmat(scale, 16, seed=seed)
    ptr, idx, deg = g.csc()
    x, info = g.pagerank(0.85, 1e-4, 20)
    g.close()
    return ptr, idx, deg, x


def _same(a, b):
    return all(np.array_equal(p, q) for p, q in zip(a, b))


def test_released_blocks_are_reused_without_trace(ctx):
    want = {(s, k): _solve(ctx, s, k) for s, k in ((16, 1), (17, 2), (15, 3))}
    n, ind, col, deg = O.rmat_csc(15, 16, seed=3)
    assert np.array_equal(want[15, 3][0], ind) and np.array_equal(want[15, 3][1], col)
    for _ in range(2):
        for s, k in ((17, 2), (15, 3), (16, 1)):
            assert _same(_solve(ctx, s, k), want[s, k])
            with pytest.raises(NwgError):  # fails half way, its blocks go back
                ctx.graph_from_edges(1 << 15, np.arange(1 << 20) % (1 << 15), np.arange(1 << 20) % (1 << 16))


def test_contexts_in_threads_and_graphs_that_outlive_them(ctx):
    import torch

    want = _solve(ctx, 16, 7)
    got = [None] * 3

    def work(q):
        c = nwgraph_amd.Context(0)
        if q:
            s = torch.cuda.Stream()
            c.set_stream(s.cuda_stream)
        for _ in range(4):
            got[q] = _solve(c, 16, 7)
        g = c.rmat(16, 16, seed=7)
        handle = c.handle
        c.set_stream(0)
        c.close()
        g.close()  # after its context
        assert handle is not None

    threads = [threading.Thread(target=work, args=(q,)) for q in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(_same(r, want) for r in got)
