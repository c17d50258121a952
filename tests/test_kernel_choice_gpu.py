"""Which kernel a call launches, where two kernels take the same shape and the faster one is
chosen by a rule on sizes: both sides of each rule's line, read from the profiler's names.
"""
from __future__ import annotations

import pytest
import torch
from launched import launched

from relation_lm import _native  # noqa: F401  (registers torch.ops.relation_lm)
from relation_lm.kernels.relation_reduce import mfma_fragments, relation_reduce_fused_seq
from relation_lm.kernels.relation_select import relation_select_packed_seq
from relation_lm.workloads import RelationConfig, select_args, selection_inputs

pytestmark = pytest.mark.gpu
ops = torch.ops.relation_lm
BF, FL = torch.bfloat16, torch.float32


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


FUSED, MLP, CHAIN = "fused_reduce_kernel", "relation_mlp_kernel", "norm_reduce"


@pytest.mark.parametrize("queries,k,d,h,r,frag,kernel", [
    (4096, 8, 512, 512, 128, True, FUSED),     # two 64-row rounds against one of 128 rows
    (3840, 5, 128, 128, 64, False, FUSED),     # 2 / 1, few columns
    (8192, 5, 128, 128, 64, True, FUSED),      # 3 / 2
    (200, 8, 128, 128, 128, False, FUSED),     # 1 / 1, one hidden chunk
    (4000, 12, 256, 256, 128, False, FUSED),   # 4 / 2
    (200, 8, 512, 128, 128, False, MLP), (200, 5, 128, 512, 64, False, MLP),
    (200, 5, 128, 512, 64, True, MLP),         # the weight's order does not choose
    (5000, 6, 512, 1024, 128, False, MLP),     # 2 / 2
    (200, 8, 576, 256, 128, False, MLP), (191, 8, 576, 256, 128, False, CHAIN)])
def test_relation_reduce_kernel(device, queries, k, d, h, r, frag, kernel):
    g = torch.Generator().manual_seed(queries + d)

    def rand(*shape):
        return torch.randn(*shape, generator=g).to(BF).to(device)

    wm, w2 = rand(h, r), rand(d, h)
    anchor = torch.zeros(1, queries, dtype=torch.int32, device=device)
    partner = torch.zeros(1, queries, k, dtype=torch.int32, device=device)
    names = launched(lambda: relation_reduce_fused_seq(
        rand(1, 64, 2 * h), rand(1, 64, r), anchor, partner, wm, mfma_fragments(w2) if frag else w2,
        rand(d), torch.zeros(1, queries, k, device=device), rand(d), rand(d),
        torch.arange(queries, device=device), 1e-5))
    assert kernel in names and not any(x in names for x in {FUSED, MLP, CHAIN} - {kernel}), names


@pytest.mark.parametrize("block,rows", [(1, 1), (2, 2), (3, 8), (8, 8), (9, 16), (16, 16), (17, 32),
                                        (32, 32), (33, 64), (64, 64), (200, 64)])
@pytest.mark.parametrize("dtype", [FL, BF])
def test_block_statistics_rows(device, block, rows, dtype):
    """A thread holds the block's rows up to the next instance, no more; the statistics are fp32
    sums in row order: n + 2 roundings of 2^-24 of sum |x| and of sum d^2 (the mean's own error
    enters the deviation's square root once)."""
    x = torch.randn(3, 4 * block, 40, generator=torch.Generator().manual_seed(block)).to(dtype)
    keys = x.to(device)
    names = launched(lambda: ops.block_statistics(keys, block))
    assert f", {rows}, " in names, names
    mean, std = ops.block_statistics(keys, block)
    torch.cuda.synchronize()
    x64 = x.double().view(3, 4, block, 40)
    want = x64.mean(2)
    dev = (x64 - want[:, :, None]).square().mean(2).sqrt()
    eps = (block + 2) * 2.0 ** -24
    tol = eps * x64.abs().mean(2)
    assert bool(((mean.double().cpu() - want).abs() <= tol).all())
    assert bool(((std.double().cpu() - dev).abs() <= eps * dev + tol).all())


@pytest.mark.parametrize("batch,queries,context,block,local,top,kernel", [
    (2, 1024, 1024, 64, 128, 4, "multi_tile_kernel"),
    (1, 512, 1024, 64, 128, 4, "::select_kernel"),       # 512 x 384 candidates
    (3, 171, 1024, 64, 128, 4, "multi_tile_kernel"),     # 513 x 384
    (1, 1024, 2048, 64, 32, 2, "::select_kernel"),       # 1024 x 160
    (1, 1, 1024, 64, 128, 4, "::select_kernel"),
    (1, 256, 4096, 64, 128, 4, "::select_kernel"),
    (1, 257, 4096, 64, 128, 4, "multi_tile_kernel"),
    (2, 300, 448, 64, 128, 4, "multi_tile_kernel"),      # over 256 candidates of a short cache
    (2, 16, 448, 64, 64, 2, "select_tile_kernel")])
def test_selection_of_few_queries(device, batch, queries, context, block, local, top, kernel):
    """Either kernel gives the bits of the same rows in fp32, which select_kernel takes."""
    cfg = RelationConfig("few", batch, context, 256, block, local, top, 8, BF, seed=queries)
    inp = selection_inputs(cfg, device=device)          # the prompt's last queries
    for name in ("anchor_query", "anchor_router_query", "partner_base"):
        inp[name] = inp[name][:, context - queries:].contiguous()
    inp["positions"] = inp["positions"][context - queries:].contiguous()
    names = launched(lambda: relation_select_packed_seq(*select_args(inp, cfg)))
    assert kernel in names, names
    wide = {k: v.float() if v.dtype == BF else v for k, v in inp.items()}
    got = relation_select_packed_seq(*select_args(inp, cfg))
    want = relation_select_packed_seq(*select_args(wide, cfg))
    torch.cuda.synchronize()
    assert all(torch.equal(g, w) for g, w in zip(got, want))
