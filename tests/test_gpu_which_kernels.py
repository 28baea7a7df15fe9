"""Which kernels a call runs: what plans, the autotuner and captured solves choose shows in their scores only
where it goes wrong, so the kernels' names are looked at (torch's profiler sees every launch of the
process, replayed graphs' too)."""
import re

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
