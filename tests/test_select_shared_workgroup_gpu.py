"""select_kernel with eight queries to a workgroup (sequence calls of more than 1024 queries in
fp32 or fp16): staged key windows that start at the first query's position whatever the order of the
others, a last workgroup with waves past the end, many partners, no block picks, fp16, caches whose
statistics are not staged.  The oracle's bits, and the bits of the same rows in calls of at most 1024
queries, which have a workgroup each.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch
from launched import launched

from oracle import select as osel
from relation_lm.kernels.relation_select import relation_select_packed_seq
from relation_lm.workloads import SELECT_ORDER, RelationConfig, select_args, selection_inputs

pytestmark = pytest.mark.gpu

NAMES = ("anchor", "anchor_score", "partner", "partner_score")
QUERY_ROWS = ("anchor_query", "anchor_router_query", "partner_base")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("context,block,local,top,k,order", [
    (128, 16, 32, 2, 8, "random"), (256, 32, 64, 0, 40, "random"), (192, 32, 40, 3, 17, "falling"),
    (256, 16, 16, 4, 5, "random"), (512, 8, 100, 6, 64, "rising")])
@pytest.mark.parametrize("strict", [False, True])
def test_eight_queries_to_a_workgroup(device, dtype, context, block, local, top, k, order, strict):
    batch, queries = 3, 403                    # 1209 queries; 403 = 50 * 8 + 3
    cfg = RelationConfig("shared", batch, context, 256, block, local, top, k, torch.float32,
                         strict_valid=strict, seed=context + k)
    inp = {n: v.to(dtype) if n.split("_")[-1] in ("query", "keys", "base", "cache") else v
           for n, v in selection_inputs(cfg).items()}
    g = torch.Generator().manual_seed(k)
    rows = torch.randint(0, context, (queries,), generator=g)
    for name in QUERY_ROWS:
        inp[name] = inp[name][:, rows].contiguous()
    pos = torch.randint(0, context, (batch, queries), generator=g)
    if order != "random":
        pos = pos.sort(dim=1, descending=order == "falling").values
    pos[1, :8] = torch.tensor([-1, -70, 0, 1, context, context + local - 2, context - 1, 3])
    inp["positions"] = pos.int()
    dev = {n: v.to(device) for n, v in inp.items()}
    names = launched(lambda: relation_select_packed_seq(*select_args(dev, cfg)))
    assert "select_kernel" in names and ("false, false>" in names or "Lb0ELb0EE" in names), names
    got = relation_select_packed_seq(*select_args(dev, cfg))
    for b in range(batch):
        row = {n: v if n.endswith(("gamma", "bias")) else v[b:b + 1].contiguous()
               for n, v in dev.items()}
        want = relation_select_packed_seq(*select_args(row, cfg))
        torch.cuda.synchronize()
        for name, x, y in zip(NAMES, got, want):
            assert torch.equal(x[b:b + 1], y), (name, b)
    host = {n: v.float().numpy() if v.is_floating_point() else v.numpy() for n, v in inp.items()}
    want = osel.relation_select_packed_seq(*[host[n] for n in SELECT_ORDER], host["positions"],
                                           local, top, k, strict)
    for name, x, y in zip(NAMES, got, want):
        assert np.array_equal(x.cpu().numpy(), y), name
