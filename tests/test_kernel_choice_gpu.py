"""Which kernel a call launches, where two kernels take the same shape and the faster one is
chosen by a rule on sizes: both sides of each rule's line, read from the profiler's names.
"""
from __future__ import annotations

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from relation_lm import _native  # noqa: F401  (registers torch.ops.relation_lm)

pytestmark = pytest.mark.gpu
ops = torch.ops.relation_lm
BF, FL = torch.bfloat16, torch.float32


def launched(call):
    """Names of the kernels one call launches."""
    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages() if "rlm::" in e.key]
    assert names
    return " ".join(names)


@pytest.mark.parametrize("m,n,k,tile", [
    (3584, 512, 192, 64), (4096, 768, 192, 64),        # 448 and 768 tiles of 64 x 64
    (3200, 1024, 192, 128), (3584, 1024, 192, 128),    # 800 and 896
    (28672, 128, 576, 64), (28672, 128, 192, 128),     # one column of 128 x 128 tiles: 896
    (33000, 128, 576, 128), (40000, 64, 576, 128),     # 256 tiles of 128 x 128 and more
    (16384, 1024, 192, 256)])
def test_linear_tile_size(device, m, n, k, tile):
    a, w = torch.ones(m, k, dtype=BF, device=device), torch.ones(n, k, dtype=BF, device=device)
    names = launched(lambda: ops.relation_linear(a, w, None, BF))
    assert "dma_tile_kernel" in names and f"{tile}, {tile}," in names, names
