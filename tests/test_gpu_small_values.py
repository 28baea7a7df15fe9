"""Scores many orders of magnitude below the others keep a float's precision: row sums in fixed point cut
bits off contributions below 2^-37 and lose those below 2^-60, so the item sweeps (nwgraph_amd/csrc/items.hip)
add such rows up once more, and the one-workgroup solves (small.hip) give way to them.

The graph is layered: mass enters at layer 0 and falls by about 10 a layer; from layers 4, 12 and 18 it
is collected in rows of 600 and of 3000 in-edges (shorter and longer than a work item).  As a DAG it holds
exact path sums after as many sweeps as it has layers.

Bounds: with u = 2^-24 a float or double row sum of m terms is within (m + 1) u, and the contributions' and
the update's roundings within 5 u, of a row's value (all terms have one sign but the adjoint's, where it is
the sum of absolute values): e' <= d A e + (m + 6) u (|b| + d A |x|), evaluated with the float64 sweeps."""
import ctypes

import numpy as np
import pytest

from nwgraph_amd import _lib

pytestmark = pytest.mark.gpu

U = 2.0**-24
LAYERS, WIDTH = 22, 8


def _layered(extra, seed):
    """edges of the graph, and how many vertices it has; extra: vertices besides"""
    rng = np.random.default_rng(seed)
    src, dst = [], []

    def link(a, b):
        src.append(np.broadcast_to(a, np.shape(b)).ravel() if np.ndim(b) else np.ravel(a))
        dst.append(np.broadcast_to(b, np.shape(a)).ravel() if np.ndim(a) and not np.ndim(b) else np.ravel(b))

    layer = np.arange(LAYERS * WIDTH).reshape(LAYERS, WIDTH)
    sinks = layer.size + np.arange(400)
    n = layer.size + sinks.size
    for l in range(LAYERS):
        for v in layer[l]:
            link(v, rng.choice(sinks, 8, replace=False))
            if l + 1 < LAYERS:
                link(v, rng.choice(layer[l + 1], 2, replace=False))
    for l, m in ((4, 600), (12, 600), (18, 600), (18, 3000)):
        if n + m + 1 + extra > 4096 and not extra:
            break
        mid = n + np.arange(m)
        link(layer[l][np.arange(m) % WIDTH], mid)
        link(mid, np.full(m, n + m))
        link(np.full(3, n + m), sinks[:3])
        n += m + 1
    if not extra:  # the one-workgroup sizes: rows of 600 only
        assert n <= 4096
    n += extra
    src, dst = np.concatenate(src), np.concatenate(dst)
    assert src.size == dst.size
    return n, src.astype(np.uint32), dst.astype(np.uint32)


def _csc(ctx, extra, seed=1):
    n, src, dst = _layered(extra, seed)
    g = ctx.graph_from_edges(n, src, dst)
    ptr, col, deg = g.csc()
    return g, n, ptr, col, deg, np.repeat(np.arange(n), np.diff(ptr.astype(np.int64)))


def _sweeps(n, to, frm, w, b, y, d, sweeps):
    m = np.bincount(to, minlength=n)
    e = np.zeros(n)
    for _ in range(sweeps):
        ay = np.abs(b) + d * np.bincount(to, weights=np.abs(w * y[frm]), minlength=n)
        e = d * np.bincount(to, weights=np.abs(w) * e[frm], minlength=n) + (m + 6) * U * ay
        y = b + d * np.bincount(to, weights=w * y[frm], minlength=n)
    return y, e


def _check(got, want, bound):
    # normal floats, so that the bound is relative
    keep = np.abs(want) > 2.0**-120
    assert np.all(np.abs(got[keep] - want[keep]) <= bound[keep])
    assert np.all(got[want == 0.0] == 0.0)


SIZES = [0, 6000]  # solved by one workgroup, and over items
D = float(np.float32(0.85))


def _teleport(n):
    v = np.zeros(n, np.float32)
    v[:WIDTH] = 1.0 / WIDTH
    return v


@pytest.mark.parametrize("how", ["as it is", "degree ordered", "timed", "in place"])
@pytest.mark.parametrize("extra", SIZES)
def test_personalised_scores(ctx, extra, how):
    g, n, ptr, col, deg, row = _csc(ctx, extra)
    if how == "degree ordered":
        g.set_plan(relabel=1)
    v = _teleport(n)
    w = 1.0 / deg[col].astype(np.float64)
    sweeps = 60
    want, e = _sweeps(n, row, col, w, (1 - D) * v.astype(np.float64), np.full(n, 1.0 / n), D, sweeps)
    assert want[want > 0].min() < 2.0**-70
    for _ in range(3):
        got, info = g.pagerank(D, 0.0, sweeps, teleport=v, kernel_timing=how == "timed", inplace=how == "in place")
        assert info["iterations"] == sweeps
        _check(got, want, e)
    # a solve that needs none of it on the same graph
    got, _ = g.pagerank(D, 0.0, 20)
    _check(got, *_sweeps(n, row, col, w, np.full(n, (1 - D) / n), np.full(n, 1.0 / n), D, 20))
    g.close()


@pytest.mark.parametrize("call", ["resident", "one call", "no alloc"])
@pytest.mark.parametrize("extra", SIZES)
def test_damping_one(ctx, extra, call):
    """Damping 1 has no base: after 17 sweeps a vertex holds what 17-edge paths brought."""
    g, n, ptr, col, deg, row = _csc(ctx, extra)
    w = 1.0 / deg[col].astype(np.float64)
    want, e = _sweeps(n, row, col, w, np.zeros(n), np.full(n, 1.0 / n), 1.0, 17)
    assert want[want > 0].min() < 2.0**-62
    if call == "resident":
        got, _ = g.pagerank(1.0, -1.0, 17)
    elif call == "one call":
        import nwgraph_amd

        got = np.zeros(n, np.float32)
        nwgraph_amd.page_rank(nwgraph_amd.Adjacency(ptr, col), deg, got, 1.0, -1.0, 17, 1, ctx=ctx)
    else:
        import torch

        dev = [torch.from_numpy(a.astype(np.int32)).cuda() for a in (ptr, col, deg)]
        x = torch.full((n,), -1.0, device="cuda")
        info = _lib.PrInfo()
        torch.cuda.synchronize()
        ctx.check(ctx.lib.nwg_pagerank_f32_noalloc(ctx.handle, n, col.size, dev[0].data_ptr(), dev[1].data_ptr(),
                                                   dev[2].data_ptr(), x.data_ptr(), 1.0, -1.0, 17,
                                                   ctypes.byref(info)))
        got = x.cpu().numpy()
    _check(got, want, e)
    g.close()


@pytest.mark.parametrize("extra", SIZES)
def test_damping_one_many_graphs(ctx, extra):
    parts = [_csc(ctx, 0, 1), _csc(ctx, extra, 2), _csc(ctx, 0, 3)]
    mg = ctx.multigraph([p[0] for p in parts])
    for _ in range(3):
        got, _, _, _ = mg.pagerank(1.0, -1.0, 17)
        for q, (g, n, ptr, col, deg, row) in enumerate(parts):
            want, e = _sweeps(n, row, col, 1.0 / deg[col].astype(np.float64), np.zeros(n), np.full(n, 1.0 / n), 1.0, 17)
            _check(got[mg.offsets[q] : mg.offsets[q + 1]], want, e)
    mg.close()
    for p in parts:
        p[0].close()


@pytest.mark.parametrize("extra", SIZES)
@pytest.mark.parametrize("scale", [1.0, 2.0**70, 2.0**-40])
def test_weighted_scores_and_gradients(ctx, extra, scale):
    """Weighted forward from a teleport at layer 0, and the adjoint of a gradient at the collecting rows and
    the sinks, which falls towards layer 0 in the same way; both scaled."""
    g, n, ptr, col, deg, row = _csc(ctx, extra)
    rng = np.random.default_rng(4)
    w = rng.uniform(0.5, 1.0, col.size).astype(np.float32)
    g.set_weights(w)
    wn = w / np.bincount(col, weights=w.astype(np.float64), minlength=n)[col]
    v = _teleport(n) * np.float32(scale)
    c = np.zeros(n, np.float32)
    c[LAYERS * WIDTH - WIDTH : LAYERS * WIDTH] = rng.normal(size=WIDTH) * scale
    sweeps = 60
    want, e = _sweeps(n, row, col, wn, (1 - D) * v.astype(np.float64), np.full(n, 1.0 / n), D, sweeps)
    lam, el = _sweeps(n, col, row, wn, c.astype(np.float64), c.astype(np.float64), D, sweeps)
    for _ in range(3):
        x, fi = g.wpr_forward(v, D, 0.0, sweeps)
        _check(x, want, e)
        _, gv, bi = g.wpr_backward(x, c, D, 0.0, sweeps, raw_weights=False)
        _check(gv, (1 - D) * lam, el + 3 * U * np.abs(lam))
        assert fi["iterations"] == bi["iterations"] == sweeps
    g.close()
