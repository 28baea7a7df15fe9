"""The builder's sort, duplicate removal and row pointers (nwgraph_amd/csrc/prims.hip, build.hip) at the
edges of their tiles: edge counts around a sort tile (4096) and a pointer tile (2048), vertex counts
at 8-bit digit boundaries, edge lists with nothing to keep, long runs of empty rows, one row, all
edges equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _want(n, src, dst, clean):
    key = dst.astype(np.uint64) * np.uint64(n) + src
    if clean:
        key = np.unique(key[src != dst])
    else:
        key = np.sort(key)
    row, col = key // np.uint64(n), (key % np.uint64(n)).astype(np.uint32)
    ptr = np.searchsorted(row, np.arange(n + 1, dtype=np.uint64)).astype(np.uint32)
    return ptr, col, np.bincount(col, minlength=n).astype(np.uint32)


@pytest.mark.parametrize("clean", [True, False])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 4096, 65537, 3000001])
@pytest.mark.parametrize("m", [1, 2, 2047, 2049, 4095, 4096, 4097, 70000])
def test_build_matches_numpy(ctx, n, m, clean):
    rng = np.random.default_rng(n + m)
    src = rng.integers(0, n, m).astype(np.uint32)
    dst = rng.integers(0, n, m).astype(np.uint32)
    src[m // 2:] = src[: m - m // 2]  # duplicates
    dst[m // 2:] = dst[: m - m // 2]
    g = ctx.graph_from_edges(n, src, dst, clean=clean)
    got = g.csc()
    assert all(np.array_equal(a, b) for a, b in zip(got, _want(n, src, dst, clean)))
    if clean and m == 4097:  # the transpose and its positions
        ptr, idx, pos = g.csr()
        row = np.repeat(np.arange(n), np.diff(got[0].astype(np.int64)))
        order = np.argsort(got[1], kind="stable")
        assert np.array_equal(pos, order) and np.array_equal(idx, row[order])
        assert np.array_equal(ptr, np.searchsorted(got[1][order], np.arange(n + 1)))
    g.close()


@pytest.mark.parametrize("kind", ["loops only", "one row", "one edge often", "last rows only", "far apart"])
def test_build_shapes(ctx, kind):
    n, m = 200000, 50000
    i = np.arange(m, dtype=np.uint32)
    src, dst = {"loops only": (i, i), "one row": (i, np.full(m, 3, np.uint32)),
                "one edge often": (np.full(m, 7, np.uint32), np.full(m, n - 1, np.uint32)),
                "last rows only": (i, n - 1 - i % 2), "far apart": (i, (i // 10000) * 49999)}[kind]
    dst = dst.astype(np.uint32)
    g = ctx.graph_from_edges(n, src, dst, clean=True)
    assert all(np.array_equal(a, b) for a, b in zip(g.csc(), _want(n, src, dst, True)))
    g.close()


@pytest.mark.parametrize("n", [1 << 22, (1 << 22) + 1])  # 256 id ranges in one pass, and one more
def test_degrees_by_range(ctx, n):
    import ctypes
    import torch
    from nwgraph_amd import DeviceGraph, _lib

    m = (1 << 24) + 3
    gen = torch.Generator(device="cuda").manual_seed(1)
    col = torch.randint(0, n, (m,), generator=gen, device="cuda", dtype=torch.int32)
    col[: m // 3] = n - 1  # a hub, whose range is split over workgroups
    col[m // 3: m // 2] %= 1000
    ptr = torch.full((n + 1,), m, device="cuda", dtype=torch.int32)
    ptr[0] = 0
    torch.cuda.synchronize()
    h = ctypes.c_void_p()
    ctx.check(ctx.lib.nwg_graph_create_csc(ctx.handle, n, m, ptr.data_ptr(), col.data_ptr(), None,
                                           _lib.NWG_MEM_DEVICE, ctypes.byref(h)))
    g = DeviceGraph(ctx, h)
    assert np.array_equal(g.csc()[2].astype(np.int64), torch.bincount(col, minlength=n).cpu().numpy())
    g.close()
