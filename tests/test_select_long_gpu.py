"""GPU parity of the sequence-form selection over longer caches and odd block counts.

relation_select_packed_seq with bf16 activations takes a matrix-core-filtered kernel
for every cache of at most 64 blocks: rlm_select_tile.hip up to 512 rows and 256
candidates, rlm_multi_tile.hip (one slot) beyond, except for few queries there, which
take select_kernel too.  The same call in fp32 runs
select_kernel (rlm_select.hip), one float64 dot per candidate; on the same values both
must give the same bits -- indices, scores, sentinels -- also for infinite, NaN and
overflowing scores, where the filter's error bound does not hold.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import select as osel
from relation_lm.kernels.relation_select import (multi_relation_select_seq,
                                                 relation_select_packed_seq)
from relation_lm.workloads import (MULTI_CONFIGS, SELECT_ORDER, RelationConfig, multi_select_args,
                                   multi_selection_inputs, select_args, selection_inputs)

pytestmark = pytest.mark.gpu

NAMES = ("anchor", "anchor_score", "partner", "partner_score")


def config(context, block, local, top, k, strict=False, batch=2, seed=1):
    return RelationConfig("long", batch, context, 256, block, local, top, k, torch.bfloat16,
                          strict_valid=strict, seed=seed)


def upcast(inp):
    return {k: v.float() if v.dtype == torch.bfloat16 else v for k, v in inp.items()}


def check_same(got, want, what):
    for name, g, w in zip(NAMES, got, want):
        assert g.shape == w.shape and g.dtype == w.dtype
        same = (g == w) | ((g != g) & (w != w))
        assert bool(same.all()), (what, name, torch.nonzero(~same)[:4].tolist(), g[~same][:4], w[~same][:4])


def check(inp, cfg, device, what):
    dev = {k: v.to(device) for k, v in inp.items()}
    got = relation_select_packed_seq(*select_args(dev, cfg))
    want = relation_select_packed_seq(*select_args(upcast(dev), cfg))
    torch.cuda.synchronize()
    check_same(got, want, what)
    return got


# Cache rows, block, local window, picks, k: over 512 rows; over 256 candidates; 7, 14,
# 11 and 3 blocks (rows of block keys padded, waves partly used); 64 blocks.
SHAPES = [(1024, 32, 64, 4, 8), (1024, 16, 32, 2, 5), (2048, 64, 128, 4, 8), (640, 64, 100, 16, 16),
          (512, 64, 128, 4, 7), (512, 32, 300, 8, 1), (448, 64, 64, 2, 8), (448, 32, 64, 4, 6),
          (176, 16, 32, 3, 8), (96, 32, 16, 1, 16), (4096, 64, 1, 2, 3)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("strict", [False, True])
def test_equals_per_query_kernel(device, shape, strict):
    cfg = config(*shape, strict=strict, seed=sum(shape) + strict)
    inp = selection_inputs(cfg, device="cpu")
    got = check(inp, cfg, device, f"{shape} strict={strict}")
    if shape[0] <= 640:
        host = {k: v.float().numpy() if v.is_floating_point() else v.numpy() for k, v in inp.items()}
        want = osel.relation_select_packed_seq(*[host[k] for k in SELECT_ORDER], host["positions"],
                                               cfg.local_window, cfg.top_blocks, cfg.k_out, strict)
        for name, g, w in zip(NAMES, got, want):
            assert np.array_equal(g.cpu().numpy(), w), (shape, name)


@pytest.mark.parametrize("shape", [(1024, 32, 64, 4, 8), (512, 64, 128, 4, 8), (448, 64, 64, 2, 8)])
def test_positions_and_ragged_queries(device, shape):
    """Positions before the first row and past the cache (with and without a candidate),
    37 queries, one position row per batch row."""
    cfg = config(*shape, seed=77)
    inp = selection_inputs(cfg, device="cpu")
    for name in ("anchor_query", "anchor_router_query", "partner_base"):
        inp[name] = inp[name][:, :37].contiguous()
    pos = torch.randint(0, shape[0], (2, 37), generator=torch.Generator().manual_seed(5))
    pos[0, :8] = torch.tensor([-1, -70, 0, 1, shape[0], shape[0] + 40, shape[0] + 4000, shape[0] - 1])
    inp["positions"] = pos.int()
    check(inp, cfg, device, f"{shape} positions")
    none = config(shape[0], shape[1], shape[2], 0, shape[4], seed=78)
    check(inp, none, device, f"{shape} no picks")


@pytest.mark.parametrize("shape", [(1024, 32, 64, 4, 8), (512, 64, 128, 4, 8), (704, 64, 100, 4, 16)])
def test_positions_and_ragged_queries_of_a_long_prompt(device, shape):
    """The same on the shared-tile kernel, which fewer queries do not reach: 2 x 1001 of them."""
    cfg = config(*shape, seed=79)
    inp = selection_inputs(cfg, device="cpu")
    g = torch.Generator().manual_seed(6)
    rows = torch.randint(0, shape[0], (1001,), generator=g)
    for name in ("anchor_query", "anchor_router_query", "partner_base"):
        inp[name] = inp[name][:, rows].contiguous()
    pos = torch.randint(0, shape[0], (2, 1001), generator=g)
    pos[0, :8] = torch.tensor([-1, -70, 0, 1, shape[0], shape[0] + 40, shape[0] + 4000, shape[0] - 1])
    pos[1, 960:976] = -5                   # a tile without any candidate
    pos[1, 990:] = shape[0] + 300
    inp["positions"] = pos.int()
    check(inp, cfg, device, f"{shape} positions")
    none = config(shape[0], shape[1], shape[2], 0, shape[4], seed=80)
    check(inp, none, device, f"{shape} no picks")


def test_equal_keys(device):
    """Every candidate ties: more members than one window, the tie rules decide."""
    cfg = config(1024, 32, 64, 4, 8, seed=9)
    inp = selection_inputs(cfg, device="cpu")
    inp["anchor_keys"][:] = inp["anchor_keys"][:, :1]
    inp["partner_keys"][0] = inp["partner_keys"][0, 7:8]
    inp["partner_keys"][1, ::2] = inp["partner_keys"][1, 3:4]
    check(inp, cfg, device, "equal keys")


@pytest.mark.parametrize("shape", [(1024, 32, 64, 4, 8), (512, 32, 300, 8, 8), (1024, 64, 128, 4, 8),
                                   (448, 64, 64, 2, 8)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3e38, -3e38])
def test_scores_that_are_not_finite(device, shape, value):
    cfg = config(*shape, seed=31)
    inp = selection_inputs(cfg, device="cpu")
    g = torch.Generator().manual_seed(2)
    rows = torch.randperm(shape[0], generator=g)[: shape[0] // 8]
    for name in ("anchor_keys", "partner_keys"):
        inp[name][0, rows, 5] = value       # one element of some rows
        inp[name][1, rows[:3]] = value      # a few whole rows
    dev = {k: v.to(device) for k, v in inp.items()}
    got = relation_select_packed_seq(*select_args(dev, cfg))
    want = relation_select_packed_seq(*select_args(upcast(dev), cfg))
    torch.cuda.synchronize()
    check_same(got, want, f"{shape} {value}")


@pytest.mark.parametrize("context,block,slots", [(320, 64, 3), (352, 32, 2), (192, 64, 4)])
def test_multi_anchor_block_counts(device, context, block, slots):
    """Block counts that are no multiple of four, through the shared-tile kernel."""
    import dataclasses

    cfg = dataclasses.replace(MULTI_CONFIGS["cfg5"], batch=2, context=context, block_size=block,
                              local_window=64, top_blocks=4, slots=slots, k_out=5, seed=context)
    inp = multi_selection_inputs(cfg, device=device)
    got = multi_relation_select_seq(*multi_select_args(inp, cfg))
    want = multi_relation_select_seq(*multi_select_args(upcast(inp), cfg))
    torch.cuda.synchronize()
    check_same(got, want, f"{context}/{block}")
    for value in (float("inf"), float("-inf")):
        wild = {k: v.clone() for k, v in inp.items()}
        for name in ("anchor_keys", "partner_keys"):
            wild[name][0, ::9, 0, 3] = value
        got = multi_relation_select_seq(*multi_select_args(wild, cfg))
        want = multi_relation_select_seq(*multi_select_args(upcast(wild), cfg))
        torch.cuda.synchronize()
        check_same(got, want, f"{context}/{block} {value}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(512, 32, 64, 4, 8), (512, 16, 32, 2, 5), (384, 64, 100, 16, 16),
                                   (448, 32, 1, 2, 3)])
@pytest.mark.parametrize("strict", [False, True])
def test_a_workgroup_per_query_gives_the_same_bits(device, dtype, shape, strict):
    """select_kernel: up to 1024 queries each have a workgroup, beyond eight share one."""
    context, block, local, top, k = shape
    cfg = config(context, block, local, top, k, strict, batch=4, seed=5)
    cast = lambda v: v.to(dtype) if v.dtype == torch.bfloat16 else v
    dev = {n: cast(v).to(device) for n, v in selection_inputs(cfg).items()}
    whole = relation_select_packed_seq(*select_args(dev, cfg))
    shared = {n: v for n, v in dev.items() if v.shape[:1] != (4,) or n.endswith(("gamma", "bias"))}
    for b in range(4):
        row = {n: v if n in shared else v[b:b + 1].contiguous() for n, v in dev.items()}
        got = relation_select_packed_seq(*select_args(row, cfg))
        torch.cuda.synchronize()
        check_same(got, [w[b:b + 1] for w in whole], (shape, b))


@pytest.mark.parametrize("shape", [(512, 32, 64, 4, 8), (256, 64, 200, 0, 4), (128, 16, 32, 2, 8)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3e38])
def test_scores_that_are_not_finite_whole_block_counts(device, shape, value):
    """The shared-tile kernel at block counts that are multiples of four."""
    test_scores_that_are_not_finite(device, shape, value)


@pytest.mark.parametrize("context,block,slots", [(320, 64, 3), (192, 64, 4), (256, 64, 3),
                                                 (512, 32, 4)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3e38])
def test_multi_anchor_scores_that_are_not_finite(device, context, block, slots, value):
    """multi_select_kernel's results, at block counts that are multiples of four and not."""
    import dataclasses

    cfg = dataclasses.replace(MULTI_CONFIGS["cfg5"], batch=2, context=context, block_size=block,
                              local_window=64, top_blocks=4, slots=slots, k_out=5, seed=context)
    inp = multi_selection_inputs(cfg, device=device)
    g = torch.Generator().manual_seed(3)
    rows = torch.randperm(context, generator=g)[: context // 8]
    for name in ("anchor_keys", "partner_keys"):
        inp[name][0, rows, 0, 3] = value          # one slot's element of some rows
        inp[name][1, rows[:3]] = value            # every slot of a few rows
        inp[name][1, rows[3:8], 1:] = value
    got = multi_relation_select_seq(*multi_select_args(inp, cfg))
    want = multi_relation_select_seq(*multi_select_args(upcast(inp), cfg))
    torch.cuda.synchronize()
    check_same(got, want, f"{context}/{block} {value}")
