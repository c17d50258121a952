"""The fused relation reduce on the 128-row kernel it is named after, at partner counts that are no
power of two (padded rows), d_model 128 to 512, relation dim 32 to 128, ragged rows, [B,Tq]
positions, indices outside the cache and queries without an active partner, against the three ops
it stands for.  relation_reduce_fused_seq sends many of these shapes to another kernel when they
have few queries, so each case checks the name of the kernel that ran: relation dim 32 and short
hidden dims stay on this one at any size, the others from a second round of 64-row tiles on.

The hidden is the same bf16 value up to the rare one on a rounding boundary (fp32 sums in another
order), worth at most 2^-8 of one of H products: 5e-3 bounds a normalised output, and the root mean
square stays below 5e-4.
"""
from __future__ import annotations

import pytest
import torch
from launched import launched

from relation_lm.kernels.relation_reduce import (mfma_fragments, relation_hidden_cached_seq,
                                                 relation_linear, relation_norm_reduce_seq,
                                                 relation_reduce_fused_seq)
from relation_lm.workloads import RelationConfig, reduce_inputs

pytestmark = pytest.mark.gpu


def check(device, batch, queries, k, d, h, r, rows=80):
    cfg = RelationConfig("fused", batch, rows, d, 16, 32, 2, k, torch.bfloat16, relation_dim=r,
                         hidden_dim=h, seed=d + h + k)
    red = reduce_inputs(cfg, device=device)
    expanded = relation_linear(red["operand_cache"], red["expanded_weight"], red["expanded_bias"])
    g = torch.Generator().manual_seed(31 * k + d)
    anchor = torch.randint(0, rows, (batch, queries), generator=g).int()
    partner = torch.randint(0, rows, (batch, queries, k), generator=g)
    score = torch.randn(batch, queries, k, generator=g)
    score[torch.rand(score.shape, generator=g) < 0.2] = -torch.inf
    score[0, 1] = -torch.inf                   # no active partner: the row is 0
    partner[0, 1] = -3                         # outside the cache: zeros
    partner[-1, 2] = rows + 5
    pos = torch.randint(0, 4 * k, (batch, queries), generator=g)  # active partners 1 to k
    a, p, s, t = anchor.to(device), partner.to(device), score.to(device), pos.int().to(device)

    def call(second):
        return relation_reduce_fused_seq(expanded, red["operand_cache"], a, p,
                                         red["product_weight"], second, red["second_bias"], s,
                                         red["norm_weight"], red["norm_bias"], t, 1e-5)

    names = launched(lambda: call(red["second_weight"]))
    assert "fused_reduce_kernel" in names, names
    got, frag = call(red["second_weight"]), call(mfma_fragments(red["second_weight"]))
    hidden = relation_hidden_cached_seq(expanded, red["operand_cache"], a, p, red["product_weight"])
    raw = relation_linear(hidden, red["second_weight"], red["second_bias"], torch.float32)
    want = relation_norm_reduce_seq(raw, s, red["norm_weight"], red["norm_bias"], t, 1e-5)
    torch.cuda.synchronize()
    off = (got - want).abs()
    assert got.shape == (batch, queries, d)
    assert float(off.max()) <= 5e-3 and float(off.square().mean().sqrt()) <= 5e-4
    assert bool((got[0, 1] == 0).all())
    assert torch.equal(frag, got)


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 7, 8, 12, 16])
@pytest.mark.parametrize("d,h,r", [(128, 128, 64), (256, 128, 128), (384, 256, 32), (512, 384, 32)])
def test_few_queries(device, k, d, h, r):
    check(device, 3, 37, k, d, h, r)


# Two 64-row rounds on 256 CUs against one of 128 rows (or three against two).
@pytest.mark.parametrize("queries,k", [(6701, 1), (2003, 3), (1401, 4), (1111, 5), (1001, 6),
                                       (835, 7), (701, 8), (667, 12), (501, 16)])
@pytest.mark.parametrize("d,h,r", [(384, 256, 64), (512, 256, 128), (256, 512, 64)])
def test_partial_rounds(device, queries, k, d, h, r):
    check(device, 3, queries, k, d, h, r)
