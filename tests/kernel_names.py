"""Names of the kernels a call runs, as torch's profiler sees them in this process."""
import collections
import re


def kernels(call):
    """{kernel name: launches} of a call, with and without its template arguments"""
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
            name = m.group(1).replace(" ", "")
            for k in {name, name.split("<")[0]}:
                names[k] += e.count
    return names
