"""Several threads with graphs of their own on one context: its calls take turns, as they share the context's
stream, events, kept memory and the host memory that solves leave their changes in."""
import threading

import numpy as np
import pytest

import nwgraph_amd

pytestmark = pytest.mark.gpu


def test_threads_on_one_context():
    c = nwgraph_amd.Context(0)
    sizes = [(300, 900), (5000, 40000), (900, 4000), (60001, 300000)]
    graphs, want = [], []

    def solve(g, w):
        x, info = g.pagerank(0.99, 1e-7, 60)
        y, fi = g.wpr_forward(None, 0.85, 1e-6, 100)
        gw, gv, bi = g.wpr_backward(y, w, 0.85, 1e-3, 100)
        return [x, y, gw, gv, info["error_trace"], fi["error_trace"], bi["error_trace"]]

    for q, (n, m) in enumerate(sizes):
        rng = np.random.default_rng(q)
        g = c.graph_from_edges(n, rng.integers(0, n, m), rng.integers(0, n, m))
        g.set_weights(rng.uniform(0.1, 1.0, g.nnz).astype(np.float32))
        graphs.append((g, rng.normal(size=n).astype(np.float32)))
        want.append(solve(*graphs[q]))
        # several segments of sweeps where few edges leave the sums (60 sweeps at most)
    assert max(w[4].size for w in want) > 28
    wrong = []

    def work(q):
        try:
            for _ in range(20):
                got = solve(*graphs[q])
                wrong.extend((q, k) for k in range(len(got)) if not np.array_equal(got[k], want[q][k]))
        except Exception as e:  # noqa: BLE001
            wrong.append((q, e))

    threads = [threading.Thread(target=work, args=(q,)) for q in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:5]
    for g, _ in graphs:
        g.close()
    c.close()
