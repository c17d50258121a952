"""GPU parity of the relation MLP kernel with the bias, LayerNorm, active-K softmax and
partner sum as its epilogue -- the form relation_reduce_fused_seq takes for d_model values
the fused kernel does not (any multiple of 32 up to 768, from 1536 rows on) and for grids its
128-row tiles fill badly -- against the three ops it stands for (relation_hidden_cached_seq,
relation_linear, relation_norm_reduce_seq).

The hidden is the same bf16 value up to the rare one on a rounding boundary (fp32 sums in
another order), worth at most 2^-8 of one of H products: 5e-3 bounds a normalised output, and
the root mean square stays below 5e-4.  Shapes: column blocks that do and do not divide among
the waves (1 to 24 of them), K that divides 64 and K that leaves padding rows, a last tile cut
short, one tile, relation dim 64 and 128, one and many hidden chunks.
"""
from __future__ import annotations

import pytest
import torch

from relation_lm.kernels.relation_reduce import (mfma_fragments, relation_hidden_cached_seq,
                                                 relation_linear, relation_norm_reduce_seq,
                                                 relation_reduce_fused_seq)
from relation_lm.workloads import RelationConfig, reduce_inputs

pytestmark = pytest.mark.gpu


def inputs(device, batch, queries, k, d, h, r, seed=0, rows=96):
    cfg = RelationConfig("mlp", batch, rows, d, 16, 32, 2, k, torch.bfloat16, relation_dim=r,
                         hidden_dim=h, seed=seed + d + h + k)
    red = reduce_inputs(cfg, device=device)
    g = torch.Generator().manual_seed(d * 31 + k)
    expanded = (red["operand_cache"].float() @ red["expanded_weight"].float().T
                + red["expanded_bias"].float()).to(torch.bfloat16)
    anchor = torch.randint(0, rows, (batch, queries), generator=g).int()
    partner = torch.randint(0, rows, (batch, queries, k), generator=g).int()
    score = torch.randn(batch, queries, k, generator=g)
    score[torch.rand(score.shape, generator=g) < 0.2] = -torch.inf
    score[0, 0] = -torch.inf                 # no active partner: the row is 0
    partner[0, 0] = -3                       # outside the cache: zeros
    pos = torch.arange(queries) * 3
    return red, expanded, anchor.to(device), partner.to(device), score.to(device), pos.to(device)


def chain(red, expanded, a, p, score, pos):
    hidden = relation_hidden_cached_seq(expanded, red["operand_cache"], a, p, red["product_weight"])
    raw = relation_linear(hidden, red["second_weight"], red["second_bias"], torch.float32)
    return relation_norm_reduce_seq(raw, score, red["norm_weight"], red["norm_bias"], pos, 1e-5)


def fused(red, expanded, a, p, score, pos):
    return relation_reduce_fused_seq(expanded, red["operand_cache"], a, p, red["product_weight"],
                                     red["second_weight"], red["second_bias"], score,
                                     red["norm_weight"], red["norm_bias"], pos, 1e-5)


@pytest.mark.parametrize("batch,queries,k,d,h,r", [
    (2, 99, 8, 576, 2304, 128), (1, 311, 5, 576, 256, 64), (3, 121, 6, 768, 384, 128),
    (2, 140, 7, 320, 128, 128), (1, 1601, 1, 32, 128, 64), (2, 49, 16, 96, 640, 128),
    (1, 130, 12, 640, 256, 64), (4, 150, 3, 224, 512, 128), (2, 130, 8, 736, 256, 128),
    (2, 71, 11, 544, 256, 128),
    # shapes the fused kernel takes too: one round of either, K = 5 and 7
    (1, 1, 8, 256, 256, 128), (2, 40, 5, 512, 512, 64), (1, 33, 7, 384, 128, 128),
    (3, 20, 16, 128, 256, 128)])
def test_equals_the_three_ops(device, batch, queries, k, d, h, r):
    args = inputs(device, batch, queries, k, d, h, r)
    got, want = fused(*args), chain(*args)
    torch.cuda.synchronize()
    off = (got - want).abs()
    assert got.shape == (batch, queries, d)
    assert float(off.max()) <= 5e-3 and float(off.square().mean().sqrt()) <= 5e-4
    assert bool((got[0, 0] == 0).all())


def test_position_and_parameter_types(device):
    red, expanded, a, p, score, pos = inputs(device, 2, 140, 6, 576, 256, 128)
    want = chain(red, expanded, a, p, score, pos)
    pos2 = pos[None].expand(2, -1).contiguous().int()
    for name in ("second_bias", "norm_weight", "norm_bias"):
        red[name] = red[name].float()
    got = fused(red, expanded, a.long(), p.long(), score, pos2)
    torch.cuda.synchronize()
    assert float((got - want).abs().max()) <= 5e-3
    again = fused(red, expanded, a.long(), p.long(), score, pos2)
    assert torch.equal(got, again)


def test_fragment_order_weight_gives_the_same_bits(device):
    args = inputs(device, 2, 40, 5, 512, 512, 64)
    want = fused(*args)
    red = dict(args[0], second_weight=mfma_fragments(args[0]["second_weight"]))
    got = fused(red, *args[1:])
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_zero_weight_rows_do_not_count(device):
    """A row beyond the active K may hold anything: its weight is 0 and it adds 0."""
    red, expanded, a, p, score, pos = inputs(device, 1, 270, 6, 576, 256, 128)
    score = torch.randn(1, 270, 6, generator=torch.Generator().manual_seed(3)).to(device)
    pos = torch.zeros(270, dtype=torch.int64, device=device)   # one active partner per query
    want = fused(red, expanded, a, p, score, pos)
    expanded = expanded.clone()
    expanded[0, 90] = float("nan")
    p = p.clone()
    a = torch.where(a == 90, 0, a).int()
    p = torch.where(p == 90, 0, p).int()
    base = fused(red, expanded, a, p, score, pos)
    p[..., 1:] = 90
    got = fused(red, expanded, a, p, score, pos)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(got).all()) and torch.equal(got, base)
    assert want.shape == got.shape


def test_long_calls_equal_their_batch_rows(device):
    """A hidden of 2.4 GB, which never exists: the call's bits are those of its batch rows."""
    red, expanded, a, p, score, pos = inputs(device, 8, 2048, 8, 64, 4608, 128, rows=512)
    got = fused(red, expanded, a, p, score, pos)
    for b in range(8):
        one = dict(red, operand_cache=red["operand_cache"][b:b + 1])
        want = fused(one, expanded[b:b + 1], a[b:b + 1], p[b:b + 1], score[b:b + 1], pos)
        torch.cuda.synchronize()
        assert torch.equal(got[b:b + 1], want), b
