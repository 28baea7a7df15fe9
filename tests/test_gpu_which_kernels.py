"""Which kernels a call runs: what plans, the autotuner and captured solves choose shows in their scores only
where it goes wrong, so the kernels' names are looked at (torch's profiler sees every launch of the
process, replayed graphs' too)."""
import re

import numpy as np
import pytest

from kernel_names import kernels

pytestmark = pytest.mark.gpu


def test_kernels_are_seen(ctx):
    g = ctx.rmat(14, 16, seed=1)
    for _ in range(3):  # launched one by one, recorded, replayed
        assert kernels(lambda: g.pagerank(0.85, -1.0, 20))["pr_item_kernel"] == 20
    g.close()


@pytest.mark.parametrize("scale", [12, 15])
def test_autotuner_times_what_it_names(ctx, scale):
    """Sizes at which a binned plan that leaves the bin size open runs the item sweep: the binned candidates'
    numbering and hints are timed with the binned kernels, and the item sweep's plan has no hints."""
    for seed in range(1, 4):
        g = ctx.rmat(scale, 16, seed=40 + seed)
        seen = kernels(g.autotune)
        for hints in (0, 1, 2):
            assert seen[f"pr_bin_kernel<false,{hints},false,13>"] >= 8  # two times four sweeps
        # numberings, hints, and the second bin size
        assert sum(c for k, c in seen.items() if re.fullmatch(r"pr_bin_kernel<false,\d,false,13>", k)) >= 6 * 8
        assert sum(c for k, c in seen.items() if re.fullmatch(r"pr_bin_kernel<false,\d,false,14>", k)) >= 8
        plan = g.get_plan()
        if not plan["binned"]:
            ran = kernels(lambda: g.pagerank(0.85, -1.0, 20))
            assert (plan["stream_hints"] == 0) or not ran["pr_item_kernel"], plan
        assert not plan["binned"] or plan["bin_bits"] in (13, 14)
        g.close()


def _graph(ctx, n, m, hub=0):
    """n vertices and exactly m edges, the first `hub` of them out-edges of vertex 7"""
    rng = np.random.default_rng(n + m)
    src, dst = rng.integers(0, n, m).astype(np.uint32), rng.integers(0, n, m).astype(np.uint32)
    src[:hub] = 7
    return ctx.graph_from_edges(n, src, dst, clean=False)


def _sweep(seen):
    return {name for name in ("small_solve_kernel", "pr_item_kernel", "pr_bin_kernel", "pr_tile_kernel")
            if any(k.split("<")[0] == name for k in seen)}


M = 1 << 20


@pytest.mark.parametrize("n,m,hub,want", [
    # one workgroup: up to 4096 rows and 20,480 edges
    (4096, 20480, 0, "small_solve_kernel"), (4097, 20480, 0, "pr_item_kernel"), (4096, 20481, 0, "pr_item_kernel"),
    # the pull plan's items below 2^18 edges, a binned plan's from there
    (30001, (1 << 18) - 1, 0, "pr_item_kernel"), (30001, 1 << 18, 0, "pr_item_kernel"),
    # below 2 M edges always; from there long rows without a hub go binned: 9 edges a row, from 3 M on 7.5
    (200001, 2 * M - 1, 0, "pr_item_kernel"), (200001, 2 * M, 0, "pr_bin_kernel"),
    (234001, 2 * M, 0, "pr_item_kernel"), (232001, 2 * M, 0, "pr_bin_kernel"),
    (200001, 2 * M, 60000, "pr_item_kernel"),
    (400001, 3 * M - 1, 0, "pr_item_kernel"), (400001, 3 * M, 0, "pr_bin_kernel"), (420001, 3 * M, 0, "pr_item_kernel"),
    # from 6.3 M edges always
    (2000001, 6 * M - 1, 0, "pr_item_kernel"), (2000001, 6 * M, 0, "pr_bin_kernel"),
    (400001, 6 * M - 1, 60000, "pr_item_kernel"), (400001, 6 * M, 60000, "pr_bin_kernel"),
])
def test_default_plan_by_size_and_degrees(ctx, n, m, hub, want):
    g = _graph(ctx, n, m, hub)
    assert g.nnz == m
    assert _sweep(kernels(lambda: g.pagerank(0.85, 1e-4, 20))) == {want}
    plan = g.get_plan()
    assert plan["binned"] == (m >= 1 << 18) and plan["bin_bits"] == 0 and plan["relabel"] == (hub > 0)
    if want != "small_solve_kernel":  # cutoffs of the plan's own ask for the row classes, a bin size for bins
        g.set_plan(binned=0, short_max=4)
        assert "pr_tile_kernel" in _sweep(kernels(lambda: g.pagerank(0.85, 1e-4, 3)))
        g.set_plan(binned=1, bin_bits=13, short_max=8)
        assert _sweep(kernels(lambda: g.pagerank(0.85, 1e-4, 3))) == {"pr_bin_kernel"}
    g.close()


@pytest.mark.parametrize("n,m,want", [(4096, 20480, "small_weighted_kernel"), (4097, 20480, "wpr_item_kernel"),
                                      (4096, 20481, "wpr_item_kernel"),
                                      # 2560 items of 1020 rows and edges
                                      (1020 * 560, 1020 * 2000, "wpr_item_kernel"),
                                      (1020 * 560 + 1, 1020 * 2000, "pr_bin_kernel")])
def test_weighted_sweep_by_size(ctx, n, m, want):
    g = _graph(ctx, n, m)
    rng = np.random.default_rng(1)
    g.set_weights(rng.uniform(0.1, 1.0, m).astype(np.float32))
    c = rng.normal(size=n).astype(np.float32)
    names = ("small_weighted_kernel", "wpr_item_kernel", "pr_bin_kernel", "wsweep_kernel")
    for call in (lambda: g.wpr_forward(None, 0.85, 1e-4, 30), lambda: g.wpr_backward(c, c, 0.85, 1e-2, 30)):
        assert {k for k in names if any(s.split("<")[0] == k for s in kernels(call))} == {want}
    g.close()


@pytest.mark.parametrize("row,look", [(12000, False), (13500, True)])  # 2^34 * 0.15 / 200,001 is 12,885
def test_small_rows_are_looked_for_where_the_base_allows_them(ctx, row, look):
    n = 200001
    rng = np.random.default_rng(row)
    src, dst = rng.integers(0, n, 3 * n).astype(np.uint32), rng.integers(0, n, 3 * n).astype(np.uint32)
    dst[:row] = 9
    g = ctx.graph_from_edges(n, src, dst, clean=False)
    form = lambda call: {k for k in kernels(call) if k.startswith(("pr_item_kernel<", "pr_item_many_kernel<"))}
    name = "pr_item_kernel<true>" if look else "pr_item_kernel<false>"
    for _ in range(2):
        assert form(lambda: g.pagerank(0.85, 1e-4, 20)) == {name}
    v = np.full(n, 1.0 / n, np.float32)
    assert form(lambda: g.pagerank(0.85, 1e-4, 20, teleport=v)) == {"pr_item_kernel<true>"}
    assert form(lambda: g.pagerank(1.0, 1e-4, 20)) == {"pr_item_kernel<true>"}
    assert form(lambda: g.pagerank(0.85, 1e-4, 20)) == {name}
    t = ctx.rmat(14, 8, seed=1)
    mg = ctx.multigraph([t, g])
    mg.set_plan(0)
    assert form(lambda: mg.pagerank(0.85, 1e-4, 20)) == {name.replace("item", "item_many")}
    assert form(lambda: mg.pagerank(1.0, 1e-4, 20)) == {"pr_item_many_kernel<true>"}
    for h in (mg, t, g):
        h.close()
