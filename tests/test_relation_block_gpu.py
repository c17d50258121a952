"""The multi-anchor block after its selection in two launches
(``relation_lm_block::relation_block_seq_out``) against the two operators it stands
for (``relation_hidden_linear_seq_out`` + ``multi_relation_reduce_seq_out``,
reference multi_relation_blocks.py:148-178).

Both make the same MLP rows bit for bit (one kernel body).  They differ in the order
of fp32 sums over the D values of a row's mean and variance, its K rows and S slots:
at most ~(D + S*K) * 2^-24 relative to the summands, which the LayerNorm keeps of
order sqrt(D) / row: a context bound of 768 * 2^-24 * 8 < 4e-4; measured far below.
The residual output adds one rounding of hidden's type.
"""

import pytest
import torch

import relation_lm  # noqa: F401
from relation_lm.kernels.relation_reduce import mfma_fragments

pytestmark = pytest.mark.gpu


def inputs(device, batch, queries, slots, k, d, h, r, dtype, seed=3):
    g = torch.Generator().manual_seed(seed)
    bf = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(device, torch.bfloat16)
    t = max(queries, 24)
    pos = torch.arange(queries) + t - queries
    pos[: min(queries, 3)] = torch.arange(min(queries, 3))       # slots past the position
    n = queries * slots
    top = pos.repeat_interleave(slots).clamp(min=0)
    a = (torch.rand(batch, n, generator=g) * (top + 1)).long().clamp(max=t - 1)
    p = (torch.rand(batch, n, k, generator=g) * (top[:, None] + 1)).long().clamp(max=t - 1)
    score = torch.randn(batch, queries, slots, k, generator=g)
    score[torch.rand(score.shape, generator=g) < 0.2] = float("-inf")
    score[:, -1, 0] = float("-inf")                               # a slot with no partner
    hidden = torch.randn(batch, queries, d, generator=g).to(device, dtype)
    return dict(
        expanded=bf(batch, t, 2 * h), operand=bf(batch, t, r), anchor=a.int().to(device),
        partner=p.int().to(device), wm=mfma_fragments(bf(h, r, scale=r ** -0.5)),
        w2=mfma_fragments(bf(d, h, scale=h ** -0.5)), b2=bf(d, scale=0.1), score=score.to(device),
        nw=(1 + 0.1 * torch.randn(d, generator=g)).to(device, dtype), nb=bf(d, scale=0.1),
        mix=torch.randn(slots, generator=g).to(device), gate=torch.tensor(0.3, device=device),
        hidden=hidden, pos=pos.to(device))


def block(v, context=True, pos=None):
    out = torch.empty_like(v["hidden"])
    ctx = torch.empty(out.shape, device=out.device) if context else None
    torch.ops.relation_lm_block.relation_block_seq_out(
        v["expanded"], v["operand"], v["anchor"], v["partner"], v["wm"], v["w2"], v["b2"],
        v["score"], v["nw"], v["nb"], v["mix"], v["gate"], v["hidden"],
        v["pos"] if pos is None else pos, 1e-5, out, ctx)
    return out, ctx


def two_ops(v):
    b, q, s, k = v["score"].shape
    d = v["hidden"].shape[-1]
    raw = torch.empty(b, q * s, k, d, device=v["score"].device)
    torch.ops.relation_lm.relation_hidden_linear_seq_out(
        v["expanded"], v["operand"], v["anchor"], v["partner"], v["wm"], v["w2"], raw)
    out = torch.empty_like(v["hidden"])
    ctx = torch.empty(out.shape, device=out.device)
    torch.ops.relation_lm.multi_relation_reduce_seq_out(
        raw.view(b, q, s, k, d), v["score"], v["nw"], v["nb"], v["mix"], v["gate"], v["hidden"],
        v["pos"], 1e-5, v["b2"], out, ctx)
    return out, ctx


# K = 5, 6, 7: groups that two 64-row tiles share; 4, 8, 16: none; 1: one row a group.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("batch, queries, slots, k, d, h, r", [
    (1, 1, 1, 1, 256, 128, 64), (1, 3, 2, 5, 256, 128, 64), (2, 37, 4, 6, 768, 256, 128),
    (1, 65, 3, 7, 512, 256, 64), (3, 16, 4, 4, 512, 128, 128), (1, 50, 8, 8, 256, 384, 128),
    (1, 29, 4, 16, 768, 128, 64), (1, 11, 2, 31, 256, 128, 64),
    (1, 9, 1, 64, 512, 128, 64), (2, 300, 2, 6, 768, 128, 128)])
def test_equals_the_two_ops(device, dtype, batch, queries, slots, k, d, h, r):
    v = inputs(device, batch, queries, slots, k, d, h, r, dtype)
    out, ctx = block(v)
    want, wctx = two_ops(v)
    alone, _ = block(v, context=False)
    pos2 = v["pos"][None].expand(batch, -1).contiguous().int()
    again, actx = block(v, pos=pos2)
    torch.cuda.synchronize()
    off = float((ctx - wctx).abs().max())
    print("largest difference", off, flush=True)
    assert off <= 4e-4
    ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -23)
    scale = torch.maximum(want.float().abs(), torch.ones((), device=device))
    assert bool(((out.float() - want.float()).abs() <= 4e-4 + ulp * scale).all())
    assert torch.equal(alone, out) and torch.equal(again, out) and torch.equal(actx, ctx)


def test_zero_weight_rows_do_not_count(device):
    v = inputs(device, 1, 40, 2, 6, 256, 128, 64, torch.bfloat16)
    live = torch.isfinite(v["score"]).view(1, 80, 6)
    spare = v["expanded"].shape[1] - 1
    v["anchor"] = torch.where(v["anchor"] == spare, 0, v["anchor"]).int()
    v["partner"] = torch.where(v["partner"] == spare, 0, v["partner"]).int()
    want, wctx = block(v)
    v["expanded"][:, spare] = float("nan")
    v["partner"] = torch.where(live, v["partner"], spare).int()
    out, ctx = block(v)
    torch.cuda.synchronize()
    assert torch.equal(out, want) and torch.equal(ctx, wctx)


def test_opcheck(device):
    v = inputs(device, 1, 7, 2, 5, 256, 128, 64, torch.bfloat16)
    out = torch.empty_like(v["hidden"])
    ctx = torch.empty(out.shape, device=device)
    torch.library.opcheck(
        torch.ops.relation_lm_block.relation_block_seq_out.default,
        (v["expanded"], v["operand"], v["anchor"], v["partner"], v["wm"], v["w2"], v["b2"],
         v["score"], v["nw"], v["nb"], v["mix"], v["gate"], v["hidden"], v["pos"], 1e-5, out, ctx))
