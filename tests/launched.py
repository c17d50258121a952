"""The kernels that a call launches, by name."""
from __future__ import annotations

import torch
from torch.profiler import ProfilerActivity, profile


def launched(call):
    """Names of the kernels one call launches (mangled where a parameter is _Float16)."""
    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages() if "rlm::" in e.key or "3rlm" in e.key]
    assert names
    return " ".join(names)
