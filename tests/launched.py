"""The kernels that a call launches, by name."""
from __future__ import annotations

import torch
from torch.profiler import ProfilerActivity, profile


def launched(call):
    """Names of the kernels one call launches (mangled where a parameter is _Float16)."""
    call()
    torch.cuda.synchronize()
    for _ in range(3):                  # a trace now and then comes back empty
        with profile(activities=[ProfilerActivity.CUDA]) as prof:
            call()
            torch.cuda.synchronize()
        names = [e.key for e in prof.key_averages() if "rlm::" in e.key or "3rlm" in e.key]
        if names:
            return " ".join(names)
    raise AssertionError("no kernel of the library in the trace")
