"""Memory that only makes a call faster is no reason to refuse it: with too little left for the sort of a union's
degree order the union keeps its numbering, and what one context keeps for later calls goes to another that
needs it.  The device's memory is taken by allocations that are never written."""
import time

import numpy as np
import pytest

import nwgraph_amd

pytestmark = pytest.mark.gpu


class _Taken:
    """All of the device's free memory but `leave` bytes."""

    def __init__(self, leave):
        import torch

        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        self.blocks = []
        for _ in range(8):  # what was freed before comes back after a while
            free, _ = torch.cuda.mem_get_info()
            if free > leave:
                self.blocks.append(torch.empty(free - leave, dtype=torch.uint8, device="cuda"))
            time.sleep(0.1)

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        import torch

        self.blocks = None
        torch.cuda.empty_cache()


def test_union_without_room_for_its_degree_order():
    c = nwgraph_amd.Context(0)
    graphs = [c.rmat(20, 16, seed=q) for q in range(3)]
    edges = sum(g.nnz for g in graphs)
    want = [g.pagerank(0.85, 1e-4, 20)[0] for g in graphs]
    c.close()  # and what it kept
    c = nwgraph_amd.Context(0)
    # the union's arrays take 4 bytes an edge, the sort 16 more, its results 4
    assert 4 * edges < 200 << 20 < 16 * edges - (500 << 20)
    with _Taken(560 << 20):
        mg = c.multigraph(graphs)
        got, its, _, _ = mg.pagerank(0.85, 1e-4, 20)
    for q, g in enumerate(graphs):
        assert np.array_equal(got[mg.offsets[q] : mg.offsets[q + 1]], want[q])
    mg.close()
    c.close()
    for g in graphs:
        g.close()


def test_memory_kept_by_another_context():
    a, b = nwgraph_amd.Context(0), nwgraph_amd.Context(0)
    m = 80 << 20
    ptr = np.full(1001, m, np.uint32)
    ptr[0] = 0
    col = np.zeros(m, np.uint32)
    with _Taken(1290 << 20):
        a.rmat(21, 16, seed=1).close()  # leaves 1130 MB of temporaries with a
        g = b.graph_from_csc(ptr, col)  # 320 MB of ids
        assert g.nnz == m and g.csc()[2][0] == m
        g.close()
    x = a.rmat(12, 16, seed=1)
    assert abs(x.pagerank()[0].sum() - 1) < 0.5
    x.close()
    a.close()
    b.close()
