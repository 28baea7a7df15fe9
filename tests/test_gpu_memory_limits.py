"""Memory that only makes a call faster is no reason to refuse it: with too little left for the sort of a union's
degree order the union keeps its numbering.  The device's memory is taken by one allocation that is
never written."""
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
        free, _ = torch.cuda.mem_get_info()
        self.block = torch.empty(free - leave, dtype=torch.uint8, device="cuda")

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        import torch

        self.block = None
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
