"""The GPU kernels that a call launches, by name."""
from collections import Counter

import pytest
import torch
from torch.profiler import ProfilerActivity, profile


def launched(call):
    """Counter of the library's kernels over call(): name with its template arguments -> launches."""
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    names = Counter()
    for e in p.key_averages():
        if "lmx::k_" in e.key:
            names[e.key.split("lmx::", 1)[1].split("(", 1)[0]] += e.count
    if not names:
        pytest.skip("no kernel records from this profiler")
    return names


def count(names, prefix):
    """Launches of the kernels whose name starts with prefix."""
    return sum(n for k, n in names.items() if k.startswith(prefix))
