"""Out-degrees counted in private 16-bit histograms (nwgraph_amd/csrc/build.hip): vertex counts at the
edges of an id range (65536 ids) and of a word (two ids), entry counts at the edges of a chunk and
of a 16-byte load, one id filling whole chunks."""
import numpy as np
import pytest

from nwgraph_amd import NwgError, _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 65535, 65536, 65537, 200003])
@pytest.mark.parametrize("m", [1, 5, 4095, 4097, 61440 * 3 + 2])
def test_counted_and_checked_degrees(ctx, n, m):
    rng = np.random.default_rng(n * 7 + m)
    col = rng.integers(0, n, m).astype(np.uint32)
    col[m // 3:] = n - 1  # one hub: runs of more than 2^16 - 1 equal ids at the largest m
    ptr = np.full(n + 1, m, np.uint32)
    ptr[0] = 0
    want = np.bincount(col, minlength=n).astype(np.uint32)
    g = ctx.graph_from_csc(ptr, col)
    assert np.array_equal(g.csc()[2], want)
    g.close()
    ctx.graph_from_csc(ptr, col, want).close()
    low = want.copy()
    low[n - 1] -= 1
    with pytest.raises(NwgError) as e:
        ctx.graph_from_csc(ptr, col, low)
    assert e.value.code == _lib.NWG_EINVAL


@pytest.mark.parametrize("what", ["entry", "descending", "end"])
def test_bad_host_csc_is_refused(ctx, what):
    n, m = 70001, 30000
    ptr = np.minimum(np.arange(n + 1), m).astype(np.uint32)
    col = (np.arange(m) % n).astype(np.uint32)
    if what == "entry":
        col[m - 1] = n
    elif what == "descending":
        ptr[5] = 9
    else:
        ptr[n] = m - 1
    with pytest.raises(NwgError) as e:
        ctx.graph_from_csc(ptr, col)
    assert e.value.code == _lib.NWG_EINVAL
