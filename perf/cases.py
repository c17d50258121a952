"""Performance cases of the routed relation path, through its public entry points.

Families (a case's ``kind``):

  decode      one token: packed cache projection with the router update, routed
              selection, relation hidden, second linear, norm-reduce, output head prep
  prefill     a prompt: expanded cache, selection and relation reduce at every position
  projection  the packed sparse-cache projection of a prompt's memory rows
  anchors     routed multi-anchor selection of one layer
  mlp         a multi-anchor layer's relation MLP and slot reduce, given the selection
  block       a whole multi-anchor relation layer

``listed`` names the configurations of ``relation_lm.workloads`` and of the
benchmark where one exists; ``draw`` varies batch, length, widths, routing, dtype
and cache form around them.
"""
from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(1, os.path.join(os.getcwd(), "relation-lm_amd"))

from relation_lm.inference import pack_sparse_cache_projection_weights  # noqa: E402
from relation_lm.kernels.relation_reduce import (  # noqa: E402
    factor_relation_first_layer,
    mfma_fragments,
    recommended_relation_cache_mode,
    relation_hidden_cache_update,
    relation_hidden_cached,
    relation_hidden_cached_seq_out,
    relation_hidden_linear_seq_fits,
    relation_hidden_linear_seq_out,
    relation_linear,
    relation_linear_out,
    relation_norm_reduce_output,
    relation_reduce_fused_seq,
    relation_reduce_fused_seq_fits,
)
from relation_lm.kernels.relation_select import (  # noqa: E402
    multi_relation_select_seq,
    relation_select_packed,
    relation_select_packed_seq,
    relation_select_packed_seq_expand,
)
from relation_lm.kernels.ring import (  # noqa: E402
    relation_hidden_cache_update_ring,
    relation_hidden_cached_ring,
    relation_select_packed_ring,
    router_cache_update_ring,
)
from relation_lm.kernels.router_cache import router_cache_update  # noqa: E402
from relation_lm.models import MultiRelationBlockConfig  # noqa: E402
from relation_lm.models.multi_relation_blocks import MultiAnchorRelationBlock  # noqa: E402
from relation_lm.workloads import SELECT_ORDER, RelationConfig, decode_step  # noqa: E402

E = 64              # exact vector width
HEADS, HEAD_DIM = 4, 16
RD = HEADS * HEAD_DIM
BUCKETS = 16
EPS = 1e-5
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # One user's next token, 512-row cache full: the smallest call, all latency.
        dict(name="decode_1", kind="decode", batch=1, rows=512, position=511, ring=False, block=32,
             local=64, top=4, k=8, d=576, hidden=2304, r=128, dtype="bf16"),
        # The same step for a small serving batch.
        dict(name="decode_8", kind="decode", batch=8, rows=512, position=511, ring=False, block=32,
             local=64, top=4, k=8, d=576, hidden=2304, r=128, dtype="bf16"),
        # A larger serving batch far past the cache length (ring caches).
        dict(name="decode_24_ring", kind="decode", batch=24, rows=512, position=4095, ring=True,
             block=32, local=64, top=4, k=8, d=576, hidden=2304, r=128, dtype="bf16"),
        # The reference's op sequence in its own data type, mid-cache, K = 6.
        dict(name="decode_4_fp32", kind="decode", batch=4, rows=512, position=300, ring=False,
             block=32, local=64, top=4, k=6, d=576, hidden=2304, r=128, dtype="fp32"),
        # A short prompt in fp32 (the smallest configuration of the workloads).
        dict(name="prefill_128_fp32", kind="prefill", batch=1, length=128, block=16, local=32,
             top=2, k=8, d=256, hidden=1024, r=128, strict=False, dtype="fp32"),
        # The benchmark's headline step.
        dict(name="prefill_512", kind="prefill", batch=8, length=512, block=32, local=64, top=4,
             k=8, d=512, hidden=512, r=128, strict=False, dtype="bf16"),
        # Long prompts, wider MLP.
        dict(name="prefill_2048", kind="prefill", batch=8, length=2048, block=64, local=128, top=4,
             k=8, d=512, hidden=1024, r=128, strict=False, dtype="bf16"),
        # The prompt that precedes the decode steps above: the decode model's widths,
        # a length that is no power of two.
        dict(name="prefill_448_d576", kind="prefill", batch=8, length=448, block=32, local=64,
             top=4, k=8, d=576, hidden=2304, r=128, strict=False, dtype="bf16"),
        # That prompt's cache rows.
        dict(name="projection_3584", kind="projection", rows=3584, d=576, dtype="bf16"),
        # Selection of one multi-anchor layer over long sequences.
        dict(name="anchors_4096", kind="anchors", batch=4, length=4096, block=64, local=128, top=8,
             slots=4, k=6, strict=False, dtype="bf16"),
        # Relation half of such a layer on one shorter sequence.
        dict(name="mlp_1024", kind="mlp", batch=1, length=1024, slots=4, k=6, d=768, hidden=3072,
             r=128, dtype="bf16"),
        # The whole layer at full size.
        dict(name="block_4096", kind="block", batch=4, length=4096, block=64, local=128, top=8,
             slots=4, k=6, d=768, r=128, dtype="bf16"),
    ]


def draw(rng):
    def log_int(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    def mostly_bf16():
        return "fp32" if rng.random() < 0.2 else "bf16"

    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "projection", "anchors",
                       "mlp", "block"])
    dtype = mostly_bf16()
    if kind == "decode":
        rows = rng.choice([256, 512])
        ring = rng.random() < 0.3
        d, hidden = rng.choice([(576, 2304), (576, 2304), (512, 1024), (256, 1024)])
        return dict(kind=kind, batch=log_int(1, 32), rows=rows,
                    position=rng.randrange(rows, 16 * rows) if ring else rng.randrange(8, rows),
                    ring=ring, block=rng.choice([16, 32, 64]), local=rng.choice([32, 64, 128]),
                    top=rng.choice([2, 4]), k=rng.randint(5, 8), d=d, hidden=hidden, r=128,
                    dtype=dtype)
    if kind == "prefill":
        block = rng.choice([16, 32, 64])
        length = block * max(2, log_int(128, 2048) // block)
        d, hidden = rng.choice([(512, 512), (512, 1024), (576, 2304), (256, 1024), (384, 512)])
        k, r = rng.randint(5, 8), rng.choice([64, 128, 128])
        most = 4e11 if dtype == "bf16" else 3e10
        batch = log_int(1, 8)
        while batch > 1 and 2 * batch * length * k * hidden * (d + r) > most:
            batch -= 1
        while length > 2 * block and 2 * batch * length * k * hidden * (d + r) > most:
            length -= block
        return dict(kind=kind, batch=batch, length=length, block=block,
                    local=rng.choice([32, 64, 128]), top=rng.choice([2, 4]), k=k, d=d,
                    hidden=hidden, r=r, strict=rng.random() < 0.3, dtype=dtype)
    if kind == "projection":
        return dict(kind=kind, rows=log_int(1, 8192), d=rng.choice([576, 576, 512, 256]),
                    dtype=dtype)
    slots, k = rng.randint(2, 4), rng.randint(4, 6)
    if kind == "anchors":
        length = 64 * max(4, log_int(256, 4096) // 64)
        return dict(kind=kind, batch=rng.randint(1, 4) if dtype == "bf16" else 1, length=length,
                    block=64 if length > 2048 else rng.choice([32, 64]),
                    local=rng.choice([64, 128]), top=rng.choice([4, 8]), slots=slots, k=k,
                    strict=rng.random() < 0.3, dtype=dtype)
    d = rng.choice([256, 512, 768])
    length = 64 * max(2, log_int(128, 2048 if dtype == "bf16" else 256) // 64)
    if kind == "mlp":
        return dict(kind=kind, batch=rng.randint(1, 2), length=length, slots=slots, k=k, d=d,
                    hidden=4 * d, r=rng.choice([64, 128]), dtype=dtype)
    return dict(kind=kind, batch=rng.randint(1, 2), length=length, block=rng.choice([32, 64]),
                local=rng.choice([64, 128]), top=rng.choice([4, 8]), slots=slots, k=k, d=d,
                r=rng.choice([64, 128]), dtype=dtype)


# --------------------------------------------------------------------------- inputs

class _Source:
    """Seeded normal draws on the GPU."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator("cuda").manual_seed(int(seed) + 1)
        self.dtype = dtype

    def normal(self, *shape, scale=1.0, shift=0.0, dtype=None):
        x = torch.randn(*shape, generator=self.g, device="cuda") * scale + shift
        return x.to(dtype or self.dtype)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda")


def _statistics(keys, block):
    """Per-block mean and biased std of router keys, [B,NB,HEADS,HEAD_DIM] fp32."""
    b, t, _ = keys.shape
    x = keys.float().view(b, t // block, block, HEADS, HEAD_DIM)
    return x.mean(2).contiguous(), x.std(2, unbiased=False).contiguous()


def _selection(src, case, batch, rows, queries, slots=None):
    """Arguments of the selection ops by name: ``queries`` None is the decode form,
    ``slots`` None the single-anchor ops."""
    q = (batch,) if queries is None else (batch, queries)
    s = () if slots is None else (slots,)
    out = {
        "anchor_query": src.normal(*q, *s, E),
        "anchor_keys": src.normal(batch, rows, *s, E),
        "anchor_router_query": src.normal(*q, RD),
        "partner_base": src.normal(*q, *s, E + RD),
        "partner_anchor_cache": src.normal(batch, rows, *s, E + RD),
        "partner_keys": src.normal(batch, rows, *s, E),
    }
    for side in ("anchor", "partner"):
        mean, std = _statistics(src.normal(batch, rows, RD), case["block"])
        out[f"{side}_block_mean"], out[f"{side}_block_std"] = mean, std
        out[f"{side}_gamma"] = src.normal(HEADS, dtype=torch.float32)
        out[f"{side}_bias"] = src.normal(HEADS, BUCKETS, dtype=torch.float32)
    return out


def _reduce_weights(src, case):
    h, d, r = case["hidden"], case["d"], case["r"]
    f32 = torch.float32
    factors = factor_relation_first_layer(src.normal(h, 4 * r, scale=(4 * r) ** -0.5, dtype=f32),
                                          src.normal(h, scale=0.01, dtype=f32), r)
    return {
        "anchor_weight": factors.anchor_weight.to(src.dtype),
        "partner_weight": factors.partner_weight.to(src.dtype),
        "first_bias": factors.first_bias.to(src.dtype),
        "product_weight": factors.product_weight.to(src.dtype),
        "expanded_weight": factors.expanded_weight.to(src.dtype),
        "expanded_bias": factors.expanded_bias.to(src.dtype),
        "second_weight": src.normal(d, h, scale=h ** -0.5),
        "second_bias": src.normal(d, scale=0.01),
        "norm_weight": src.normal(d, scale=0.05, shift=1.0),
        "norm_bias": src.normal(d, scale=0.01),
    }


def _packed_projection(src, d):
    return pack_sparse_cache_projection_weights(
        [src.normal(w, d, scale=d ** -0.5) for w in (64, 64, 128, 128, 64, 64)])


def _prepare_decode(case, src):
    b, t, d = case["batch"], case["rows"], case["d"]
    cfg = RelationConfig("decode", b, t, d, case["block"], case["local"], case["top"], case["k"],
                         src.dtype, relation_dim=case["r"], hidden_dim=case["hidden"])
    sel = _selection(src, case, b, t, None)
    sel["position"] = torch.tensor(case["position"], dtype=torch.int64, device="cuda")
    red = _reduce_weights(src, case)
    red["operand_cache"] = src.normal(b, t, case["r"])
    router = {}
    for side in ("anchor", "partner"):
        router[f"{side}_raw_cache"] = src.normal(b, t, RD, dtype=torch.float32)
        router[f"{side}_conv_cache"] = src.normal(b, t, RD, dtype=torch.float32)
        router[f"{side}_conv_weight"] = src.normal(RD, 3, scale=0.1, dtype=torch.float32)
    expanded = (red["operand_cache"].float() @ red["expanded_weight"].float().T
                + red["expanded_bias"].float()).to(src.dtype)
    return {"cfg": cfg, "sel": sel, "red": red, "router": router, "expanded_cache": expanded,
            "memory": src.normal(b, d), "projection": _packed_projection(src, d),
            "ring": case["ring"],
            "head": {"query": src.normal(b, d), "mix": torch.tensor(-1.0, device="cuda"),
                     "weight": src.normal(d, scale=0.1, shift=1.0), "bias": src.normal(d, scale=0.1)}}


def _prepare_prefill(case, src):
    b, t = case["batch"], case["length"]
    red = _reduce_weights(src, case)
    red["operand_cache"] = src.normal(b, t, case["r"])
    st = {"sel": _selection(src, case, b, t, t), "red": red,
          "positions": torch.arange(t, device="cuda"),
          "expanded_cache": torch.empty(b, t, 2 * case["hidden"], dtype=src.dtype, device="cuda")}
    # The second weight as the fused reduce likes it best, where it takes it at all.
    w2 = red["second_weight"]
    if src.dtype == torch.bfloat16 and case["d"] % 32 == 0 and case["hidden"] % 16 == 0:
        frags = mfma_fragments(w2)
        partner = torch.empty(b, t, case["k"], dtype=torch.int32, device="cuda")
        if relation_reduce_fused_seq_fits(st["expanded_cache"], red["operand_cache"], partner,
                                          red["product_weight"], frags):
            w2 = frags
    st["second"] = w2
    return st


def _prepare_mlp(case, src):
    b, t, s, k = case["batch"], case["length"], case["slots"], case["k"]
    red = _reduce_weights(src, case)
    position = torch.arange(t, device="cuda")[None, :, None]
    op = src.normal(b, t, case["r"])
    expanded = (op.float() @ red["expanded_weight"].float().T
                + red["expanded_bias"].float()).to(src.dtype)
    anchor = (src.uniform(b, t, s) * (position + 1)).long()
    partner = (src.uniform(b, t, s, k) * (position[..., None] + 1)).long()
    score = src.normal(b, t, s, k, dtype=torch.float32)
    # The first positions have fewer candidates than partners.
    score = torch.where(torch.arange(k, device="cuda") < position[..., None] - s + 1, score,
                        torch.full_like(score, -math.inf))
    st = {"red": red, "operand_cache": op, "expanded_cache": expanded,
          "anchor": anchor.int().view(b, t * s), "partner": partner.int().view(b, t * s, k),
          "score": score, "positions": torch.arange(t, device="cuda"),
          "slot_mix": src.normal(s, dtype=torch.float32),
          "gate": torch.tensor(-1.5, device="cuda"), "stream": src.normal(b, t, case["d"]),
          "shape": (b, t, s, k, case["d"]), "fused": False}
    if src.dtype == torch.bfloat16:
        wm, w2 = mfma_fragments(red["product_weight"]), mfma_fragments(red["second_weight"])
        if relation_hidden_linear_seq_fits(expanded, op, wm, w2):
            st.update(fused=True, product=wm, second=w2)
    return st


def _prepare_block(case, src):
    cfg = MultiRelationBlockConfig(
        d_model=case["d"], gate_dim=E, relation_dim=case["r"], anchors_per_block=case["slots"],
        partners_per_anchor=case["k"], block_size=case["block"], local_window=case["local"],
        top_blocks=case["top"])
    with torch.device("cuda"):
        block = MultiAnchorRelationBlock(cfg)
    with torch.no_grad():
        for name, p in block.named_parameters():
            if name in ("residual_gate", "slot_mix_logits"):
                continue
            if "router_gamma" in name or "router_bias" in name:
                p.copy_(src.normal(*p.shape, dtype=torch.float32))
            elif p.dim() == 2:
                p.copy_(src.normal(*p.shape, scale=p.shape[1] ** -0.5, dtype=torch.float32))
            else:
                norm_weight = name in ("input_norm.weight", "relation_mlp.3.weight")
                p.copy_(src.normal(*p.shape, scale=0.05, shift=1.0 if norm_weight else 0.0,
                                   dtype=torch.float32))
    block = block.to(src.dtype).eval().requires_grad_(False)
    shape = (case["batch"], case["length"], case["d"])
    return {"block": block, "stream": src.normal(*shape), "memory": src.normal(*shape)}


def prepare(case, seed):
    src = _Source(seed, DTYPES[case["dtype"]])
    kind = case["kind"]
    if kind == "decode":
        st = _prepare_decode(case, src)
    elif kind == "prefill":
        st = _prepare_prefill(case, src)
    elif kind == "projection":
        st = {"memory": src.normal(case["rows"], case["d"]),
              "projection": _packed_projection(src, case["d"])}
    elif kind == "anchors":
        st = {"sel": _selection(src, case, case["batch"], case["length"], case["length"],
                                case["slots"]),
              "positions": torch.arange(case["length"], device="cuda")}
    elif kind == "mlp":
        st = _prepare_mlp(case, src)
    else:
        st = _prepare_block(case, src)
    st["case"] = case
    return st


# --------------------------------------------------------------------------- the calls

def _decode_fp32(st):
    """The reference's op sequence (decode_step's fused forms take bf16 caches)."""
    sel, red, rc, head, cfg = st["sel"], st["red"], st["router"], st["head"], st["cfg"]
    ring, position, expanded = st["ring"], sel["position"], st["expanded_cache"]
    row = st["case"]["position"] % cfg.context
    parts = st["projection"].project(st["memory"])
    for cache, part in zip((sel["anchor_keys"], sel["partner_keys"], red["operand_cache"],
                            sel["partner_anchor_cache"]), parts):
        cache[:, row] = part
    update_router = router_cache_update_ring if ring else router_cache_update
    update_router(parts[4], parts[5], rc["anchor_raw_cache"], rc["partner_raw_cache"],
                  rc["anchor_conv_cache"], rc["partner_conv_cache"], sel["anchor_block_mean"],
                  sel["anchor_block_std"], sel["partner_block_mean"], sel["partner_block_std"],
                  rc["anchor_conv_weight"], rc["partner_conv_weight"], position, cfg.block_size)
    select = relation_select_packed_ring if ring else relation_select_packed
    a, s, p, ps = select(*(sel[n] for n in SELECT_ORDER), position, cfg.local_window,
                         cfg.top_blocks, cfg.k_out, cfg.strict_valid)
    if recommended_relation_cache_mode(cfg.batch) == "fused_update":
        update = relation_hidden_cache_update_ring if ring else relation_hidden_cache_update
        hidden = update(expanded, red["operand_cache"], a, p, red["anchor_weight"],
                        red["partner_weight"], red["product_weight"], red["first_bias"], position)
    else:
        relation_linear_out(red["operand_cache"][:, row], red["expanded_weight"],
                            red["expanded_bias"], expanded[:, row])
        cached = relation_hidden_cached_ring if ring else relation_hidden_cached
        hidden = cached(expanded, red["operand_cache"], a, p, red["product_weight"])
    raw = relation_linear(hidden, red["second_weight"], red["second_bias"], torch.float32)
    context, final = relation_norm_reduce_output(
        raw, ps, red["norm_weight"], red["norm_bias"], position, EPS, head["query"], head["mix"],
        head["weight"], head["bias"], EPS)
    return a, s, p, ps, context, final


def _run_decode(st):
    out = (decode_step(st, st["cfg"]) if st["case"]["dtype"] == "bf16" else _decode_fp32(st))
    sel, red, rc = st["sel"], st["red"], st["router"]
    return {
        "anchor": out[0], "anchor_score": out[1], "partner": out[2], "partner_score": out[3],
        "context": out[4], "final": out[5],
        "anchor_keys": sel["anchor_keys"], "partner_keys": sel["partner_keys"],
        "operand_cache": red["operand_cache"], "partner_anchor_cache": sel["partner_anchor_cache"],
        "expanded_cache": st["expanded_cache"],
        **{n: rc[n] for n in ("anchor_raw_cache", "partner_raw_cache", "anchor_conv_cache",
                              "partner_conv_cache")},
        **{n: sel[n] for n in ("anchor_block_mean", "anchor_block_std", "partner_block_mean",
                               "partner_block_std")},
    }


def _run_prefill(st):
    case, sel, red, expanded = st["case"], st["sel"], st["red"], st["expanded_cache"]
    args = tuple(sel[n] for n in SELECT_ORDER) + (st["positions"], case["local"], case["top"],
                                                  case["k"], case["strict"])
    if case["dtype"] == "bf16":
        a, s, p, ps = relation_select_packed_seq_expand(
            *args, red["operand_cache"], red["expanded_weight"], red["expanded_bias"], expanded)
    else:
        expanded = relation_linear(red["operand_cache"], red["expanded_weight"],
                                   red["expanded_bias"])
        a, s, p, ps = relation_select_packed_seq(*args)
    context = relation_reduce_fused_seq(
        expanded, red["operand_cache"], a, p, red["product_weight"], st["second"],
        red["second_bias"], ps, red["norm_weight"], red["norm_bias"], st["positions"], EPS)
    return {"anchor": a, "anchor_score": s, "partner": p, "partner_score": ps,
            "expanded_cache": expanded, "context": context}


def _run_mlp(st):
    b, t, s, k, d = st["shape"]
    red = st["red"]
    if st["fused"]:
        raw = torch.empty(b, t * s, k, d, dtype=torch.float32, device="cuda")
        relation_hidden_linear_seq_out(st["expanded_cache"], st["operand_cache"], st["anchor"],
                                       st["partner"], st["product"], st["second"], raw)
        bias = red["second_bias"]
    else:
        hidden = torch.empty(b, t * s, k, red["second_weight"].shape[1],
                             dtype=red["second_weight"].dtype, device="cuda")
        relation_hidden_cached_seq_out(st["expanded_cache"], st["operand_cache"], st["anchor"],
                                       st["partner"], red["product_weight"], hidden)
        raw = relation_linear(hidden, red["second_weight"], red["second_bias"], torch.float32)
        bias = None
    output = torch.empty_like(st["stream"])
    context = torch.empty(b, t, d, dtype=torch.float32, device="cuda")
    torch.ops.relation_lm.multi_relation_reduce_seq_out(
        raw.view(b, t, s, k, d), st["score"], red["norm_weight"], red["norm_bias"], st["slot_mix"],
        st["gate"], st["stream"], st["positions"], EPS, bias, output, context)
    return {"output": output, "context": context}


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "decode":
        return _run_decode(st)
    if kind == "prefill":
        return _run_prefill(st)
    if kind == "projection":
        return st["projection"].project(st["memory"])
    if kind == "anchors":
        return multi_relation_select_seq(*(st["sel"][n] for n in SELECT_ORDER), st["positions"],
                                         case["local"], case["top"], case["k"], case["strict"])
    if kind == "mlp":
        return _run_mlp(st)
    return st["block"](st["stream"], st["memory"])


# --------------------------------------------------------------------------- what it takes

def _select_work(case, batch, rows, queries, slots, elem):
    """Bytes and operations of a selection: queries, keys and caches once, statistics,
    outputs; one dot per candidate and the per-block router dots."""
    nb, k = rows // case["block"], case["k"]
    n = batch * queries
    per_query = elem * (slots * E + RD + slots * (E + RD)) + 8 * slots * (1 + k)
    per_row = elem * slots * (2 * E + E + RD)
    size = n * per_query + batch * rows * per_row + 4 * batch * nb * 4 * RD
    candidates = min(rows, case["local"] + case["top"] * case["block"])
    return size, n * slots * 2 * (2 * E * candidates) + n * (1 + slots) * nb * 4 * RD


def work(case):
    elem = 2 if case["dtype"] == "bf16" else 4
    kind = case["kind"]
    if kind == "projection":
        n, d = case["rows"], case["d"]
        return {"bytes": elem * (n * d + 512 * d + n * 512), "flops": 2.0 * n * d * 512}
    if kind == "anchors":
        size, flops = _select_work(case, case["batch"], case["length"], case["length"],
                                   case["slots"], elem)
        return {"bytes": size, "flops": float(flops)}
    if kind == "decode":
        # The keys of the candidates, the gathered cache rows, every weight, the
        # token's rows; the caches beyond those need not be touched.
        b, d, h, r, k = (case[n] for n in ("batch", "d", "hidden", "r", "k"))
        nb = case["rows"] // case["block"]
        candidates = min(case["rows"], case["local"] + case["top"] * case["block"])
        weights = elem * (512 * d + 2 * h * r + h * r + h * d)
        per_query = (elem * (2 * d + 2 * E * candidates + 3 * E + RD + 2 * (E + RD) + (k + 1) * (h + r)
                             + 512 + 2 * h + d) + 4 * (4 * nb * RD + 2 * case["block"] * RD + d))
        flops = 2.0 * b * (512 * d + 2 * h * r + k * h * (r + d) + 2 * E * candidates + 4 * nb * RD)
        return {"bytes": weights + b * per_query, "flops": flops}
    b, t, d, r, k = (case[n] for n in ("batch", "length", "d", "r", "k"))
    if kind == "prefill":
        h = case["hidden"]
        size, flops = _select_work(case, b, t, t, 1, elem)
        size += elem * (b * t * (r + 2 * h) + 3 * h * r + h * d) + 4 * b * t * d
        flops += 2.0 * b * t * (2 * h * r + k * h * (r + d))
        return {"bytes": size, "flops": flops}
    s = case["slots"]
    h = case["hidden"] if kind == "mlp" else 4 * d
    size = elem * (b * t * (r + 2 * h + 2 * d) + h * r + h * d) + 4 * b * t * s * (1 + 2 * k)
    flops = 2.0 * b * t * s * k * h * (r + d)
    if kind == "mlp":
        return {"bytes": size + 4 * b * t * d, "flops": flops}
    # The whole layer: stream and memory in, output and the selection out, the weights;
    # projections of both, expanded cache, selection and relation MLP.
    widths = s * E + RD + s * (E + RD) + 2 * s * E + s * (E + RD) + 2 * RD + r
    _, select_flops = _select_work(case, b, t, t, s, elem)
    size = elem * (3 * b * t * d + widths * d + 3 * h * r + h * d) + b * t * s * (4 + 9 * k)
    return {"bytes": size, "flops": flops + select_flops + 2.0 * b * t * (widths * d + 2 * h * r)}


def tolerance(case):
    """About four times what the path differs by from 64 bits, or (block) from itself with
    the projections' sums in another order, over the listed cases and a few drawn ones."""
    kind = case["kind"]
    if kind == "anchors":
        # Indices and fp32 scores are those of float64 dots rounded once.
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    # A rounding step in a projection moves scores, and rarely a pick, of what is
    # selected from it; a prompt's selection has none before it.
    differ = 0.0 if kind == "prefill" else 5e-4
    if case["dtype"] == "fp32":
        # Seen: 4.5e-7, largest 2.2e-6 (sums of up to 2304 products).
        return {"rel": 2e-6, "max": 1e-5, "differ": differ}
    if kind == "block":
        # Seen: 1.3e-4, largest 0.024, 2e-5 of the picks.
        return {"rel": 1e-3, "max": 0.1, "differ": differ}
    # Seen: 1.7e-3 (one bf16 rounding), largest 0.010.
    return {"rel": 7e-3, "max": 0.04, "differ": differ}


# --------------------------------------------------------------------------- in 64 bits

def _f64(x):
    return x.double()


def _block_scores(query, mean, std, gamma, bias, age):
    """Router scores [Q,NB]: query [Q,RD], statistics [NB,HEADS,HEAD_DIM], age [Q,NB] the
    distance from each block's end."""
    q = _f64(query).view(-1, HEADS, HEAD_DIM)
    dots = torch.einsum("qhd,nhd->qhn", q, _f64(mean))
    spread = torch.einsum("qhd,nhd->qhn", q.abs(), _f64(std))
    bucket = torch.log2(age.clamp(min=0).double() + 1).floor().long().clamp(max=BUCKETS - 1)
    per_head = (dots + torch.log1p(torch.exp(_f64(gamma)))[None, :, None] * spread) / HEAD_DIM ** 0.5
    per_head = per_head + _f64(bias)[:, bucket].permute(1, 0, 2)
    return torch.logsumexp(per_head, dim=1).float()


def _candidates(query, mean, std, gamma, bias, t, case, rows, ring):
    """Mask [Q,rows] of the cache rows a query may take, and the rows' positions."""
    block = case["block"]
    row = torch.arange(rows, device="cuda")
    slot = torch.arange(rows // block, device="cuda")
    t = t[:, None]
    if ring:
        pos = t - torch.remainder(t - row, rows)
        number = t // block - torch.remainder(t // block - slot, rows // block)
    else:
        pos, number = row.expand(t.shape[0], -1), slot.expand(t.shape[0], -1)
    end = (number + 1) * block - 1
    start = (t - case["local"] + 1).clamp(min=0)
    eligible = (end <= t) & (number >= 0)
    if case.get("strict"):
        eligible &= end < start
    score = _block_scores(query, mean, std, gamma, bias, t - end)
    score = score.masked_fill(~eligible, -math.inf)
    top = min(case["top"], slot.numel())
    best = score.topk(top, dim=1)
    picked = torch.zeros_like(score, dtype=torch.bool).scatter_(1, best.indices,
                                                                best.values > -1e30)
    live = (pos >= 0) & (pos <= t)
    remote = picked.repeat_interleave(block, dim=1) & (pos < start)
    return live & ((pos >= start) | remote), pos


def _select64(sel, b, t, case, rows, slots, ring=False):
    """One batch row's selection for queries at positions t [Q]: (anchor [Q,S], its score,
    partner [Q,S,K], its score), positions and float64 scores."""
    def query(name):
        x = sel[name][b]
        return x.view(t.numel(), *((slots,) if name != "anchor_router_query" else ()), -1)

    def keys(name):
        return sel[name][b].view(rows, slots, -1)

    stats = {side: tuple(sel[f"{side}_{n}"][b] if n.startswith("block") else sel[f"{side}_{n}"]
                         for n in ("block_mean", "block_std", "gamma", "bias"))
             for side in ("anchor", "partner")}
    free, pos = _candidates(query("anchor_router_query"), *stats["anchor"], t, case, rows, ring)
    free = free.clone()
    anchors, anchor_scores = [], []
    for s in range(slots):
        x = (_f64(query("anchor_query")[:, s]) @ _f64(keys("anchor_keys")[:, s]).T / E ** 0.5).float()
        best = x.masked_fill(~free, -math.inf).max(dim=1)
        on = (t >= s) if slots > 1 else torch.ones_like(t, dtype=torch.bool)
        anchors.append(torch.where(on, best.indices, 0))
        anchor_scores.append(best.values.masked_fill(~on, -math.inf))
        free[torch.nonzero(on)[:, 0], best.indices[on]] = False
    taken = torch.zeros_like(free)
    for s, a in enumerate(anchors):
        on = (t >= s) if slots > 1 else torch.ones_like(t, dtype=torch.bool)
        taken[torch.nonzero(on)[:, 0], a[on]] = True
    partners, partner_scores = [], []
    for s in range(slots):
        on = (t >= s) if slots > 1 else torch.ones_like(t, dtype=torch.bool)
        row = keys("partner_anchor_cache")[:, s][anchors[s]].float()
        both = query("partner_base")[:, s].float() + row
        mask, _ = _candidates(both[:, E:], *stats["partner"], t, case, rows, ring)
        mask = mask & ~taken & on[:, None]
        x = (_f64(both[:, :E]) @ _f64(keys("partner_keys")[:, s]).T / E ** 0.5).float()
        best = x.masked_fill(~mask, -math.inf).topk(case["k"], dim=1)
        index = pos.gather(1, best.indices)
        partners.append(torch.where(best.values > -math.inf, index, (t - case["local"] + 1)[:, None]))
        partner_scores.append(best.values)
    anchor = pos.gather(1, torch.stack(anchors, 1))
    return (anchor, torch.stack(anchor_scores, 1).double(), torch.stack(partners, 1),
            torch.stack(partner_scores, 1).double())


def _gather64(cache, index):
    ok = (index >= 0) & (index < cache.shape[0])
    return _f64(cache)[index.clamp(0, cache.shape[0] - 1)] * ok[..., None]


def _raw64(expanded, operand, anchor, partner, red):
    """Second-linear rows [Q,K,D] of one batch row: expanded and operand its caches."""
    h = red["product_weight"].shape[0]
    pair = _gather64(operand, anchor)[:, None] * _gather64(operand, partner)
    pre = (pair @ _f64(red["product_weight"]).T + _gather64(expanded, anchor)[:, None, :h]
           + _gather64(expanded, partner)[..., h:])
    return F.gelu(pre) @ _f64(red["second_weight"]).T + _f64(red["second_bias"])


def _norm64(x, weight, bias):
    return F.layer_norm(x, x.shape[-1:], _f64(weight), _f64(bias), EPS)


def _context64(raw, score, t, red):
    """Active-K softmax and weighted sum of the normed rows."""
    k = score.shape[-1]
    limit = torch.ceil(torch.log2(t.double() + 2)).clamp(1, k)
    active = (torch.arange(k, device="cuda") < limit[:, None]) & (score > -1e30)
    weight = torch.softmax(torch.where(active, score, -1e4), -1) * active
    weight = weight / weight.sum(-1, keepdim=True).clamp(min=1e-9)
    return (weight[..., None] * _norm64(raw, red["norm_weight"], red["norm_bias"])).sum(1)


def _exact_decode(st, case):
    sel, red, rc, head = st["sel"], st["red"], st["router"], st["head"]
    b, rows, t = case["batch"], case["rows"], case["position"]
    at, dtype = t % rows, DTYPES[case["dtype"]]
    packed = (_f64(st["memory"]) @ _f64(st["projection"].weight).T).to(dtype)
    parts = packed.split(st["projection"].split_sizes, dim=-1)
    for cache, part in zip((sel["anchor_keys"], sel["partner_keys"], red["operand_cache"],
                            sel["partner_anchor_cache"]), parts):
        cache[:, at] = part
    out = {}
    block, j = case["block"], (t // case["block"]) % (rows // case["block"])
    for side, part in (("anchor", parts[4]), ("partner", parts[5])):
        raw, conv = _f64(rc[f"{side}_raw_cache"]), _f64(rc[f"{side}_conv_cache"])
        w = _f64(rc[f"{side}_conv_weight"])
        raw[:, at] = _f64(part)
        conv[:, at] = sum(raw[:, (t - i) % rows] * w[:, 2 - i] for i in range(3) if t >= i)
        held = conv[:, j * block:(j + 1) * block]
        if case["ring"]:  # rows past t still hold positions of the last lap
            held = held * (torch.arange(block, device="cuda") <= t % block)[:, None]
        mean, std = _f64(sel[f"{side}_block_mean"]), _f64(sel[f"{side}_block_std"])
        mean[:, j] = held.mean(1).view(b, HEADS, HEAD_DIM)
        std[:, j] = held.std(1, unbiased=False).view(b, HEADS, HEAD_DIM)
        sel[f"{side}_block_mean"], sel[f"{side}_block_std"] = mean, std
        out.update({f"{side}_raw_cache": raw, f"{side}_conv_cache": conv,
                    f"{side}_block_mean": mean, f"{side}_block_std": std})
    expanded = st["expanded_cache"]
    expanded[:, at] = (_f64(red["operand_cache"][:, at]) @ _f64(red["expanded_weight"]).T
                       + _f64(red["expanded_bias"])).to(dtype)
    position = torch.tensor([t], device="cuda")
    found = [_select64(sel, i, position, case, rows, 1, case["ring"]) for i in range(b)]
    context = torch.stack([
        _context64(_raw64(expanded[i], red["operand_cache"][i], a[:, 0] % rows, p[:, 0] % rows, red),
                   ps[:, 0], position, red)[0] for i, (a, _, p, ps) in enumerate(found)])
    mixed = _f64(head["query"]) + torch.sigmoid(_f64(head["mix"])) * context
    out.update(anchor=None, anchor_score=torch.stack([f[1][0, 0] for f in found]), partner=None,
               partner_score=torch.stack([f[3][0, 0] for f in found]), context=context,
               final=_norm64(mixed, head["weight"], head["bias"]),
               anchor_keys=_f64(sel["anchor_keys"]), partner_keys=_f64(sel["partner_keys"]),
               operand_cache=_f64(red["operand_cache"]),
               partner_anchor_cache=_f64(sel["partner_anchor_cache"]),
               expanded_cache=_f64(expanded))
    return out


def _exact_prefill(st, case):
    red, sel, t = st["red"], st["sel"], st["positions"]
    b, length = case["batch"], case["length"]
    op = red["operand_cache"]
    expanded = (_f64(op) @ _f64(red["expanded_weight"]).T + _f64(red["expanded_bias"])).to(op.dtype)
    scores, partner_scores, contexts = [], [], []
    for i in range(b):
        a, s, p, ps = _select64(sel, i, t, case, length, 1)
        a, s, p, ps = a[:, 0], s[:, 0], p[:, 0], ps[:, 0]
        contexts.append(torch.cat([
            _context64(_raw64(expanded[i], op[i], a[n:n + 256], p[n:n + 256], red), ps[n:n + 256],
                       t[n:n + 256], red) for n in range(0, length, 256)]))
        scores.append(s)
        partner_scores.append(ps)
    return {"anchor": None, "anchor_score": torch.stack(scores), "partner": None,
            "partner_score": torch.stack(partner_scores), "expanded_cache": _f64(expanded),
            "context": torch.stack(contexts)}


def _exact_mlp(st, case):
    b, t, s, k, d = st["shape"]
    red = st["red"]
    mix = torch.softmax(_f64(st["slot_mix"]), 0)
    on = torch.arange(s, device="cuda") <= st["positions"][:, None]
    mix = mix * on
    mix = mix / mix.sum(-1, keepdim=True).clamp(min=1e-9)
    context = torch.empty(b, t, d, dtype=torch.float64, device="cuda")
    for i in range(b):
        for n in range(0, t, 64):
            rows = slice(n * s, (n + 64) * s)
            raw = _raw64(st["expanded_cache"][i], st["operand_cache"][i], st["anchor"][i, rows].long(),
                         st["partner"][i, rows].long(), red)
            score = _f64(st["score"][i, n:n + 64])
            active = torch.isfinite(score)
            w = torch.softmax(torch.where(active, score, -1e4), -1) * active
            w = w / w.sum(-1, keepdim=True).clamp(min=1e-9)
            rel = _norm64(raw, red["norm_weight"], red["norm_bias"]).view(-1, s, k, d)
            context[i, n:n + 64] = torch.einsum("qs,qsk,qskd->qd", mix[n:n + 64], w, rel)
    return {"output": _f64(st["stream"]) + torch.sigmoid(_f64(st["gate"])) * context,
            "context": context}


def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        return None  # its selection follows the projections' 16-bit roundings
    st = prepare(case, seed)
    if kind == "decode":
        return _exact_decode(st, case)
    if kind == "prefill":
        return _exact_prefill(st, case)
    if kind == "mlp":
        return _exact_mlp(st, case)
    if kind == "projection":
        p = st["projection"]
        return (_f64(st["memory"]) @ _f64(p.weight).T).split(p.split_sizes, dim=-1)
    found = [_select64(st["sel"], i, st["positions"], case, case["length"], case["slots"])
             for i in range(case["batch"])]
    return (None, torch.stack([f[1] for f in found]), None, torch.stack([f[3] for f in found]))
