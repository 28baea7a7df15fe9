"""The work that programs have this library do, as measurable cases.

Each case is one call (or one training step) through the public entry points: the resident
PageRank solve, the reference-shaped one-call page_rank on host arrays, the allocation-free
call, batched personalised PageRank, the many-graphs solve, the weighted solve with its
implicit adjoint, and the graph builder.  Graphs are made from seeded random edges on the
device: RMAT (A/B/C/D = .57/.19/.19/.05, any vertex count), uniform random, and the 4-neighbour
lattice with long-range edges.
"""
import ctypes
import functools
import math
import random

import numpy as np
import torch

import nwgraph_amd
from nwgraph_amd import _lib
from nwgraph_amd.autograd import weighted_pagerank

DAMPING, TOL = 0.85, 1e-4
RMAT = (0.57, 0.19, 0.19, 0.05)


def listed():
    return [
        # a small resident graph solved again and again (latency: launches and their gaps)
        dict(name="solve_rmat12", kind="solve", graph="rmat", n=1 << 12, ef=16, teleport=False, max_iters=20),
        # the reference's CPU-sized benchmark graph, resident
        dict(name="solve_rmat16", kind="solve", graph="rmat", n=1 << 16, ef=16, teleport=False, max_iters=20),
        # personalised solve of an ordinary graph of ragged size without hubs
        dict(name="solve_urand_1500007", kind="solve", graph="urand", n=1500007, ef=16, teleport=True, max_iters=20),
        # the headline benchmark graph
        dict(name="solve_rmat25", kind="solve", graph="rmat", n=1 << 25, ef=16, teleport=False, max_iters=20),
        # a road-like graph: low degrees, high locality, more sweeps
        dict(name="solve_grid4096", kind="solve", graph="grid", n=4096 * 4096, ef=2, teleport=False, max_iters=100),
        # the drop-in page_rank(graph, degrees, scores, ...) on host containers, as the reference is called
        dict(name="dropin_200003", kind="dropin", graph="rmat", n=200003, ef=16, max_iters=20),
        # the allocation-free call of a serving loop on a CSC already in device memory
        dict(name="noalloc_100003", kind="noalloc", graph="rmat", n=100003, ef=16, max_iters=20),
        # the batched benchmark: 64 personalised vectors of 8 seeds, degree-ordered plan, tuned k-tile
        dict(name="ppr_rmat22_k64", kind="ppr", graph="rmat", n=1 << 22, ef=16, k=64, tuned=True, max_iters=20),
        # many independent graphs of mixed sizes solved in one call
        dict(name="multi_256", kind="multi", graphs=256, lo=10, hi=18, ef=16, max_iters=20),
        # weighted PageRank and its implicit adjoint, the weights resident: forward, then the gradients of c . x
        dict(name="wpr_rmat20", kind="wpr", graph="rmat", n=1 << 20, ef=16, max_iters=100),
        # a training step on a small graph through autograd: new edge weights, forward, adjoint
        dict(name="train_12007", kind="train", graph="rmat", n=12007, ef=16, max_iters=100),
        # an edge list on the device cleaned and built into a CSC with out-degrees
        dict(name="build_rmat22", kind="build", graph="rmat", n=1 << 22, ef=16),
    ]


def _log_size(rng, lo, hi):
    """An integer in [lo, hi], even over the logarithm; usually odd, now and then a power of two."""
    n = int(round(2.0 ** rng.uniform(math.log2(lo), math.log2(hi))))
    if rng.random() < 0.15:
        return min(hi, max(lo, 1 << (n.bit_length() - 1)))
    return min(hi, max(lo, n | 1))


def draw(rng):
    kind = rng.choice(["solve", "solve", "dropin", "noalloc", "ppr", "multi", "wpr", "train", "build"])
    graph = rng.choice(["rmat", "rmat", "urand"])
    ef = rng.randint(4, 24)
    if kind == "solve":
        if rng.random() < 0.2:
            w = _log_size(rng, 64, 4096)
            return dict(kind=kind, graph="grid", n=w * w, ef=2, teleport=False, max_iters=100)
        return dict(kind=kind, graph=graph, n=_log_size(rng, 1 << 10, 1 << 24), ef=ef, teleport=rng.random() < 0.3,
                    max_iters=20)
    if kind == "dropin":
        return dict(kind=kind, graph=graph, n=_log_size(rng, 1 << 8, 1 << 19), ef=ef, max_iters=20)
    if kind == "noalloc":
        return dict(kind=kind, graph=graph, n=_log_size(rng, 1 << 8, 1 << 20), ef=ef, max_iters=20)
    if kind == "ppr":
        return dict(kind=kind, graph=graph, n=_log_size(rng, 1 << 12, 1 << 20), ef=ef, k=rng.randint(1, 64),
                    tuned=rng.random() < 0.5, max_iters=20)
    if kind == "multi":
        lo = rng.randint(8, 12)
        return dict(kind=kind, graphs=rng.randint(3, 96), lo=lo, hi=lo + rng.randint(0, 6), ef=ef, max_iters=20)
    if kind == "wpr":
        return dict(kind=kind, graph=graph, n=_log_size(rng, 1 << 10, 1 << 20), ef=rng.randint(4, 16), max_iters=100)
    if kind == "train":
        return dict(kind=kind, graph=graph, n=_log_size(rng, 1 << 8, 15000), ef=rng.randint(4, 16), max_iters=100)
    return dict(kind="build", graph=graph, n=_log_size(rng, 1 << 10, 1 << 22), ef=rng.randint(4, 16))


# ------------------------------------------------------------------------------ inputs
def _edges(case, seed):
    """Raw directed edges (src, dst) as int32 device tensors, duplicates and self-loops included."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n, m = case["n"], case["ef"] * case["n"]
    if case["graph"] == "urand":
        e = torch.randint(0, n, (2, m), generator=gen, device="cuda", dtype=torch.int32)
        return e[0], e[1]
    if case["graph"] == "grid":
        w = math.isqrt(n)
        v = torch.arange(n, device="cuda", dtype=torch.int32)
        right, down = v[v % w != w - 1], v[: n - w]
        right = right[torch.rand(right.numel(), generator=gen, device="cuda") < 0.85]
        down = down[torch.rand(down.numel(), generator=gen, device="cuda") < 0.85]
        far = v[torch.rand(n, generator=gen, device="cuda") < 0.005]
        to = torch.randint(0, n, (far.numel(),), generator=gen, device="cuda", dtype=torch.int32)
        return (torch.cat([right, right + 1, down, down + w, far]), torch.cat([right + 1, right, down + w, down, to]))
    scale = max(1, (n - 1).bit_length())
    src = torch.empty(m, dtype=torch.int32, device="cuda")
    dst = torch.empty(m, dtype=torch.int32, device="cuda")
    a, b, c, _ = RMAT
    piece = 1 << 26
    for i in range(0, m, piece):
        u, v = src[i:i + piece], dst[i:i + piece]
        u.zero_()
        v.zero_()
        r = torch.empty(u.numel(), device="cuda")
        for _ in range(scale):
            r.uniform_(generator=gen)
            u.mul_(2).add_(r >= a + b)
            v.mul_(2).add_(((r >= a) & (r < a + b)) | (r >= a + b + c))
        if n != 1 << scale:  # spread the 2^scale ids over n
            u.copy_((u.to(torch.int64) * n) >> scale)
            v.copy_((v.to(torch.int64) * n) >> scale)
    return src, dst


@functools.lru_cache(maxsize=None)
def _context():
    return nwgraph_amd.Context(0)


def _build(n, src, dst):
    """The builder on edges in device memory."""
    ctx = _context()
    h = ctypes.c_void_p()
    ctx.check(ctx.lib.nwg_graph_build_from_edges(ctx.handle, n, src.numel(), ctypes.c_void_p(src.data_ptr()),
                                                 ctypes.c_void_p(dst.data_ptr()), 1, _lib.NWG_MEM_DEVICE,
                                                 ctypes.byref(h)))
    return nwgraph_amd.DeviceGraph(ctx, h)


class _DeviceArray:
    """uint32 device memory of a graph, as the array interface torch reads (every value is below 2^31)."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<i4", data=(ptr, False), version=2)


def _csc_tensors(g):
    """Copies of a graph's CSC and out-degrees that outlive it."""
    ptr, idx, deg = g.device_csc()
    out = [torch.empty(m, dtype=torch.int32, device="cuda") for m in (g.n + 1, g.nnz, g.n)]
    for t, p in zip(out, (ptr, idx, deg)):
        t.copy_(torch.as_tensor(_DeviceArray(p, t.numel()), device="cuda"))
    return out  # destroying the graph waits for the device


def _multi_cases(case):
    scales = [case["lo"] + q % (case["hi"] - case["lo"] + 1) for q in range(case["graphs"])]
    return [dict(graph="rmat", n=1 << s, ef=case["ef"]) for s in scales]


def _teleport(n, seed):
    v = torch.rand(n, generator=torch.Generator(device="cuda").manual_seed(seed + 1), device="cuda") + 0.1
    return (v.double() / v.double().sum()).float()


def _weights(n, nnz, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed + 2)
    w = 0.1 + 0.9 * torch.rand(nnz, generator=gen, device="cuda")
    return w, torch.randn(n, generator=gen, device="cuda")


def _seeds(case, seed):
    rng = np.random.default_rng(seed)
    return [rng.choice(case["n"], 8, replace=False).astype(np.uint32) for _ in range(case["k"])]


def _case_edges(case, seed):
    """The case's edges for a seed.  The weighted cases' gradients and the built CSC are as long
    as there are distinct edges, so those kinds keep one structure: the weighted cases draw new
    weights, teleports and gradients, the builder's edges are renamed by a rotation of the ids."""
    if case["kind"] not in ("wpr", "train", "build"):
        return _edges(case, seed)
    src, dst = _edges(case, 1)
    if case["kind"] == "build":
        n, by = case["n"], random.Random(seed).randrange(case["n"])
        for t in (src, dst):
            t.sub_(n - by)  # in [-n, n): no overflow
            t.add_((t < 0).to(torch.int32) * n)
    return src, dst


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, case=case)
    if kind == "multi":
        graphs = [_build(c["n"], *_edges(c, seed * 1000 + q)) for q, c in enumerate(_multi_cases(case))]
        s["mg"] = _context().multigraph(graphs)
        s["mg"].autotune()
        s["out"] = torch.empty(s["mg"].n, device="cuda")
        return s
    src, dst = _case_edges(case, seed)
    torch.cuda.synchronize()
    if kind == "build":
        s.update(src=src, dst=dst)
        return s
    g = _build(case["n"], src, dst)
    del src, dst
    if kind == "solve":
        g.set_plan()  # the plan a first solve would make
        s.update(g=g, out=torch.empty(g.n, device="cuda"), v=_teleport(g.n, seed) if case["teleport"] else None)
    elif kind == "dropin":
        ptr, idx, deg = g.csc()
        s.update(adj=nwgraph_amd.Adjacency(ptr, idx), deg=deg, out=np.zeros(g.n, np.float32))
    elif kind == "noalloc":
        s.update(csc=_csc_tensors(g), out=torch.empty(g.n, device="cuda"))
        torch.cuda.synchronize()
    elif kind == "ppr":
        seeds = _seeds(case, seed)
        if case["tuned"]:
            g.set_plan(relabel=1)
            g.ppr_autotune(seeds)
        s.update(g=g, seeds=seeds, out=torch.empty(g.n, case["k"], device="cuda"))
    else:
        w, c = _weights(g.n, g.nnz, seed)
        v = _teleport(g.n, seed)
        if kind == "train":
            s.update(g=g, w=w.requires_grad_(), v=v.requires_grad_(), c=c)
        else:
            torch.cuda.synchronize()
            g.set_weights_device(w.data_ptr())
            s.update(g=g, v=v, c=c, x=torch.empty_like(v), gw=torch.empty_like(w), gv=torch.empty_like(v))
    return s


# ------------------------------------------------------------------------------ one pass
def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "solve":
        v = s["v"]
        info = s["g"].pagerank_device(s["out"].data_ptr(), None if v is None else v.data_ptr(), DAMPING, TOL,
                                      case["max_iters"])
        return dict(scores=s["out"], iterations=info["iterations"])
    if kind == "dropin":
        info = {}
        nwgraph_amd.page_rank(s["adj"], s["deg"], s["out"], DAMPING, TOL, case["max_iters"], 1, info=info)
        return dict(scores=s["out"], iterations=info["iterations"])
    if kind == "noalloc":
        ctx, info = _context(), _lib.PrInfo()
        ptr, idx, deg = s["csc"]
        ctx.check(ctx.lib.nwg_pagerank_f32_noalloc(ctx.handle, s["out"].numel(), idx.numel(), ptr.data_ptr(),
                                                   idx.data_ptr(), deg.data_ptr(), s["out"].data_ptr(), DAMPING, TOL,
                                                   case["max_iters"], ctypes.byref(info)))
        return dict(scores=s["out"], iterations=int(info.iterations))
    if kind == "ppr":
        its, _ = s["g"].ppr_device(s["seeds"], s["out"].data_ptr(), DAMPING, TOL, case["max_iters"])
        return dict(scores=s["out"], iterations=its.astype(np.int64))
    if kind == "multi":
        ctx, mg, info = _context(), s["mg"], _lib.PrInfo()
        its = np.zeros(mg.ngraphs, np.uint64)
        ctx.check(ctx.lib.nwg_multigraph_pagerank(ctx.handle, mg.handle, s["out"].data_ptr(), DAMPING, TOL,
                                                  case["max_iters"], _lib.NWG_MEM_DEVICE, its.ctypes.data, None,
                                                  ctypes.byref(info)))
        return dict(scores=s["out"], iterations=its.astype(np.int64))
    if kind == "wpr":
        g, x, c, it = s["g"], s["x"].data_ptr(), s["c"].data_ptr(), case["max_iters"]
        g.wpr_forward_device(s["v"].data_ptr(), x, DAMPING, TOL, it, relative=True)
        g.wpr_backward_device(x, c, s["gw"].data_ptr(), s["gv"].data_ptr(), DAMPING, TOL, it, relative=True)
        return dict(x=s["x"], grad_w=s["gw"], grad_v=s["gv"])
    if kind == "train":
        s["w"].grad = s["v"].grad = None
        x = weighted_pagerank(s["w"], s["v"], s["g"], DAMPING, TOL, case["max_iters"], relative=True)
        x.backward(s["c"])
        return dict(x=x.detach(), grad_w=s["w"].grad, grad_v=s["v"].grad)
    g = _build(case["n"], s["src"], s["dst"])
    ptr, idx, deg = _csc_tensors(g)
    g.close()
    return dict(ptr=ptr, idx=idx, deg=deg)


# ------------------------------------------------------------------------------ least work
@functools.lru_cache(maxsize=None)
def _distinct(graph, n, ef):
    """Expected edges left after duplicates and self-loops are removed."""
    if graph == "grid":
        return 4 * 0.85 * n + 0.005 * n
    m = float(ef) * n
    if graph == "urand":
        return n * (n - 1.0) * -math.expm1(-m / (float(n) * n))
    # cells of the 2^s x 2^s matrix grouped by how many of their s quadrant picks were A, B, C, D
    s = max(1, (n - 1).bit_length())
    la, lb, lc, ld = (math.log(p) for p in RMAT)
    f, tot = math.lgamma, 0.0
    for i in range(s + 1):
        for j in range(s - i + 1):
            for k in range(s - i - j + 1):
                q = s - i - j - k
                logp = i * la + j * lb + k * lc + q * ld
                cells = math.exp(f(s + 1) - f(i + 1) - f(j + 1) - f(k + 1) - f(q + 1))
                if j == k == 0:
                    continue  # the diagonal
                tot += cells * -math.expm1(-m * math.exp(logp))
    return tot


def _sweeps(case):
    """Sweeps to the tolerance: RMAT uses all 20; uniform random graphs and the lattice stop earlier."""
    return min(case["max_iters"], {"rmat": 20, "urand": 7, "grid": 29}[case.get("graph", "rmat")])


def work(case):
    kind = case["kind"]
    if kind == "multi":
        return dict(bytes=sum(_sweeps(case) * (4 * _distinct("rmat", c["n"], c["ef"]) + 24 * c["n"])
                              for c in _multi_cases(case)),
                    flops=sum(_sweeps(case) * _distinct("rmat", c["n"], c["ef"]) for c in _multi_cases(case)))
    n, e = case["n"], _distinct(case["graph"], case["n"], case["ef"])
    if kind == "build":  # the edges in, the CSC and the out-degrees out
        return dict(bytes=8.0 * case["ef"] * n + 4 * e + 8 * n, flops=0)
    k = _sweeps(case)
    if kind == "ppr":  # ids, row pointers and degrees once a sweep; four k-vectors per row
        return dict(bytes=k * (4 * e + 8 * n + 16.0 * n * case["k"]), flops=k * 2.0 * e * case["k"])
    if kind in ("wpr", "train"):  # 23 forward and 14 adjoint sweeps, the edge gradient; train: the weights in
        return dict(bytes=37 * (8 * e + 16 * n) + 12 * e + 12 * n + (8 * e if kind == "train" else 0),
                    flops=37 * 2 * e + 3 * e)
    # ids, row pointers, contributions in and out, scores in and out, degrees
    return dict(bytes=k * (4 * e + 24.0 * n), flops=k * e)


# ------------------------------------------------------------------------------ in 64 bits
def _clean(n, src, dst):
    """The distinct edges without self-loops in CSC order (by target, then source), as int64."""
    key = dst.to(torch.int64) * n + src.to(torch.int64)
    key = torch.unique(key[src != dst])
    return key % n, torch.div(key, n, rounding_mode="floor")


def _offsets(ids, n):
    """Where each of the ids 0 .. n starts in an ascending list of ids."""
    return torch.searchsorted(ids, torch.arange(n + 1, device="cuda"))


def _sums(values, off):
    """Sums of values[off[i]:off[i + 1]] as differences of a running sum."""
    c = torch.cat([values.new_zeros(1), torch.cumsum(values, 0)])
    return c[off[1:]] - c[off[:-1]]


def _jacobi(n, src, dst, base, iters, groups=None, init=None):
    """PageRank sweeps in float64 -> (scores, sweeps of each group); groups ascend."""
    deg = torch.bincount(src, minlength=n).double()
    rows = _offsets(dst, n)
    group = torch.zeros(n, dtype=torch.int64, device="cuda") if groups is None else groups
    ng = int(group[-1]) + 1
    goff = _offsets(group, ng)
    x = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda") if init is None else init
    live = torch.ones(ng, dtype=torch.bool, device="cuda")
    its = torch.zeros(ng, dtype=torch.int64, device="cuda")
    for _ in range(iters):
        xn = torch.where(live[group], base + DAMPING * _sums((x / deg)[src], rows), x)
        err = _sums((xn - x).abs(), goff)
        its += live
        x, live = xn, live & (err >= TOL)
        if not bool(live.any()):
            break
    return x, its


def exact(case, seed):
    kind = case["kind"]
    if kind == "build":
        return None  # whole numbers only
    if kind == "multi":
        cs, ss, dd, gg, off = _multi_cases(case), [], [], [], 0
        for q, c in enumerate(cs):
            a, b = _clean(c["n"], *_edges(c, seed * 1000 + q))
            ss.append(a + off)
            dd.append(b + off)
            gg.append(torch.full((c["n"],), q, dtype=torch.int64, device="cuda"))
            off += c["n"]
        g = torch.cat(gg)
        size = torch.tensor([float(c["n"]) for c in cs], dtype=torch.float64, device="cuda")[g]
        x, _ = _jacobi(off, torch.cat(ss), torch.cat(dd), (1 - DAMPING) / size, case["max_iters"], g, 1 / size)
        return dict(scores=x, iterations=None)
    n = case["n"]
    src, dst = _clean(n, *_case_edges(case, seed))
    if kind in ("solve", "dropin", "noalloc"):
        base = (1 - DAMPING) * (_teleport(n, seed).double() if case.get("teleport") else 1.0 / n)
        x, _ = _jacobi(n, src, dst, base, case["max_iters"])
        return dict(scores=x.cpu().numpy() if kind == "dropin" else x, iterations=None)
    if kind == "ppr":
        return dict(scores=_ppr_exact(case, seed, src, dst), iterations=None)
    # wpr, train: x = (1-d) v + d A x, lambda = c + d A^T lambda, and the gradients of c . x
    w32, c = _weights(n, src.numel(), seed)
    w, c, v = w32.double(), c.double(), _teleport(n, seed).double()
    order = torch.argsort(src, stable=True)
    rows, outs = _offsets(dst, n), _offsets(src[order], n)
    total = _sums(w[order], outs)
    wn = w / total[src]

    def fixed_point(x, b, pull, scale):
        for _ in range(case["max_iters"]):
            xn = b + DAMPING * pull(x)
            err = float((xn - x).abs().sum())
            x = xn
            if err < TOL * scale:
                break
        return x

    x = fixed_point(torch.full_like(v, 1.0 / n), (1 - DAMPING) * v, lambda x: _sums(wn * x[src], rows), float(v.sum()))
    lam = fixed_point(c, c, lambda y: _sums((wn * y[dst])[order], outs), float(c.abs().sum()) / (1 - DAMPING))
    gw = DAMPING * lam[dst] * x[src]
    gw = (gw - _sums((gw * wn)[order], outs)[src]) / total[src]
    return dict(x=x, grad_w=gw, grad_v=(1 - DAMPING) * lam)


def _ppr_exact(case, seed, src, dst):
    n, k = case["n"], case["k"]
    deg = torch.bincount(src, minlength=n).double()[:, None]
    base = torch.zeros(n, k, dtype=torch.float64, device="cuda")
    for j, s in enumerate(_seeds(case, seed)):
        base[torch.from_numpy(s.astype(np.int64)).cuda(), j] = (1 - DAMPING) / s.size
    # rows in pieces of at most 256 in-edges, so that no sum is one long serial chain
    off = _offsets(dst, n)
    pieces = (off[1:] - off[:-1] + 255) // 256
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), pieces)
    nth = torch.arange(row.numel(), device="cuda") - (torch.cumsum(pieces, 0) - pieces)[row]
    start = off[row] + 256 * nth
    x = torch.full((n, k), 1.0 / n, dtype=torch.float64, device="cuda")
    live = torch.ones(k, dtype=torch.bool, device="cuda")
    for _ in range(case["max_iters"]):
        part = torch.nn.functional.embedding_bag(src, x / deg, start, mode="sum")
        z = torch.zeros_like(x).index_add_(0, row, part)
        xn = torch.where(live, base + DAMPING * z, x)
        err = (xn - x).abs().sum(0)
        x, live = xn, live & (err >= TOL)
        if not bool(live.any()):
            break
    return x
