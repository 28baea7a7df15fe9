"""What a call that fails leaves behind on the context's stream."""
import ctypes

import numpy as np
import pytest

import nwgraph_amd
from nwgraph_amd import _lib

pytestmark = pytest.mark.gpu


def test_refused_arguments_leave_a_recording_alone():
    """A call refused for its arguments while the caller records a HIP graph on the context's stream does not
    touch the stream: the recording goes on, and replays what was recorded."""
    import torch

    c = nwgraph_amd.Context(0)
    g = c.graph_from_csc(np.array([0, 1, 2], np.uint32), np.array([1, 0], np.uint32))
    s = torch.cuda.Stream()
    y = torch.zeros(1000, device="cuda")
    scores = torch.zeros(2, device="cuda")
    torch.cuda.synchronize()
    c.set_stream(s.cuda_stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s, capture_error_mode="thread_local"):
        y.add_(1.0)
        rc = c.lib.nwg_graph_pagerank(c.handle, g.handle, ctypes.c_void_p(scores.data_ptr()), None, 0.85, 1e-4, 20,
                                      7, None)  # no such kind of memory
        y.mul_(2.0)
    assert rc == _lib.NWG_EINVAL
    for want in (2.0, 6.0, 14.0):
        graph.replay()
        torch.cuda.synchronize()
        assert np.all(y.cpu().numpy() == want)
    x, _ = g.pagerank()
    assert np.allclose(x, 0.5)
    c.set_stream(0)
    g.close()
    c.close()
