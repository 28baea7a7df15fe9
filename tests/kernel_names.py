"""Names of the kernels a call runs, as torch's profiler sees them in this process."""
import collections
import re


def kernels(call):
    """{kernel name with template arguments: launches} of a call"""
    import torch
    from torch.profiler import ProfilerActivity, profile

    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    names = collections.Counter()
    for e in p.key_averages():
        m = re.search(r"nwg::\(anonymous namespace\)::(\w+(<[^(]*>)?)\(", e.key)
        if m:
            names[m.group(1).replace(" ", "")] += e.count
    return names
