"""Performance cases of the attention library: the work its users have it do, through the operators of
``dscuda_amd.harness.ops``.

A case is a dict of plain values.  ``op`` names the path a user's program takes:

===================  ============================================================================================
flash_forward        causal (grouped-query) attention forward, head size 64 or 128
flash_train          its forward and backward, as one training step runs them
prefill_forward      per-head MLA prefill forward, 128 + 64 columns of query and key, 128 of value
prefill_train        its forward and backward
decode               absorbed MLA decode of one query token per sequence over a paged latent cache
decode_layer         what one MLA layer runs around that decode: W_UK absorb, rotary embedding, decode with the
                     plan all layers of a step share, W_UV un-absorb
absorbed_layer       absorbed MLA prefill between its two projections: absorb, forward, un-absorb
absorbed_train       absorbed MLA forward and backward
===================  ============================================================================================

Shapes are those of the harness's suites, of the benchmark and of the tests, or lie between them.  Buffers that a
program keeps from step to step (outputs, gradients, workspaces, the decode plan, weights) are made by ``prepare``.
"""

from __future__ import annotations

import math

import torch

from dscuda_amd.harness import configs, ops

RANK, ROPE, NOPE, VALUE = configs.MLA_RANK, configs.MLA_ROPE, 128, 128
PAGE = 64
SPLITS = 8


def listed():
    return [
        # One short sequence of eight heads of 64 columns: the benchmark's flash-attention workload.  Latency.
        {"name": "flash_forward_short", "op": "flash_forward", "batch": 1, "tokens": 512, "heads": 8, "kv_heads": 8, "dim": 64},
        # Grouped-query prefill of a small batch: the largest grouped shape of the harness's full suite.
        {"name": "flash_forward_grouped", "op": "flash_forward", "batch": 4, "tokens": 2048, "heads": 8, "kv_heads": 2, "dim": 128},
        # Training step of a grouped-query layer with 64-column heads; the length is no power of two.
        {"name": "flash_train_grouped", "op": "flash_train", "batch": 2, "tokens": 1088, "heads": 16, "kv_heads": 4, "dim": 64},
        # Two short prompts of a ragged length on a few heads: the harness's ragged MLA shape.  Latency.
        {"name": "prefill_ragged", "op": "prefill_forward", "batch": 2, "tokens": 257, "heads": 4},
        # Long-context prefill with all 128 heads on one GPU: the benchmark's longest forward.
        {"name": "prefill_longest", "op": "prefill_forward", "batch": 1, "tokens": 16384, "heads": 128},
        # Training step of an eighth of the heads (one rank of a head-sharded layer), a length between the tile sizes.
        {"name": "prefill_train_shard", "op": "prefill_train", "batch": 1, "tokens": 1000, "heads": 16},
        # Training step at the benchmark's headline shape.
        {"name": "prefill_train_full", "op": "prefill_train", "batch": 1, "tokens": 4096, "heads": 128},
        # The benchmark's decode: 64 sequences of 1024 to 8192 cached tokens, 128 heads.
        {"name": "decode_batch", "op": "decode", "batch": 64, "low": 1024, "high": 8192, "heads": 128},
        # One layer of a decode step on one rank of a head-sharded server: 16 heads, 16 sequences.
        {"name": "decode_layer_shard", "op": "decode_layer", "batch": 16, "low": 1024, "high": 4096, "heads": 16},
        # Prefill of one prompt through the absorbed form with the projections on either side, 128 heads.
        {"name": "absorbed_layer", "op": "absorbed_layer", "batch": 1, "tokens": 1024, "heads": 128},
        # Training step of the absorbed form on a short sequence: the largest MLA shape of the harness's full suite.
        {"name": "absorbed_train_short", "op": "absorbed_train", "batch": 1, "tokens": 512, "heads": 8},
        # The same with all 128 heads at a usual training length.
        {"name": "absorbed_train_full", "op": "absorbed_train", "batch": 1, "tokens": 2048, "heads": 128},
    ]


# A drawn case asks for no more than these: the arithmetic and traffic of the largest listed ones.
MOST_FLOPS = {"forward": 8e12, "train": 2.4e12}
MOST_BYTES = 1.5e9


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    while True:
        op = rng.choice(["flash_forward", "flash_train", "prefill_forward", "prefill_train", "decode", "decode_layer",
                         "absorbed_layer", "absorbed_train"])
        if op in ("flash_forward", "flash_train"):
            kv_heads = rng.choice([1, 2, 4, 8])
            case = {"op": op, "batch": rng.choice([1, 1, 2, 3, 4, 8]), "tokens": 64 * _log_uniform(rng, 2, 128),
                    "heads": kv_heads * rng.choice([1, 2, 4, 8]), "kv_heads": kv_heads, "dim": rng.choice([64, 128])}
        elif op in ("prefill_forward", "prefill_train"):
            case = {"op": op, "batch": rng.choice([1, 1, 2, 3]), "tokens": _log_uniform(rng, 100, 12000),
                    "heads": rng.choice([4, 8, 16, 32, 64, 128])}
        elif op in ("decode", "decode_layer"):
            high = _log_uniform(rng, 200, 8192)
            case = {"op": op, "batch": _log_uniform(rng, 1, 64), "low": max(1, high // rng.choice([1, 2, 8])), "high": high,
                    "heads": rng.choice([8, 16, 16, 32, 64, 128])}
        else:
            case = {"op": op, "batch": rng.choice([1, 1, 2, 3]), "tokens": _log_uniform(rng, 100, 4096),
                    "heads": rng.choice([4, 8, 16, 32, 64, 128])}
        needs = work(case)
        if needs["flops"] <= MOST_FLOPS["train" if op.endswith("train") else "forward"] and needs["bytes"] <= MOST_BYTES:
            return case


# ---- what a user's program has in hand before the call --------------------------------------------------------

def prepare(case, seed):
    generator = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape, factor):
        return torch.randn(shape, device="cuda", generator=generator).mul_(factor).bfloat16()

    def empty(*shape, dtype=torch.bfloat16):
        return torch.empty(shape, device="cuda", dtype=dtype)

    op, batch, heads = case["op"], case["batch"], case["heads"]
    state = {"op": op}
    if op in ("flash_forward", "flash_train"):
        tokens, kv_heads, dim = case["tokens"], case["kv_heads"], case["dim"]
        state["scale"] = configs.c_float(dim ** -0.5)
        state["query"] = randn(batch, tokens, heads, dim, factor=1.0)
        state["key"] = randn(batch, tokens, kv_heads, dim, factor=1.0)
        state["value"] = randn(batch, tokens, kv_heads, dim, factor=1.0)
        state["out"] = torch.empty_like(state["query"])
        state["lse"] = empty(batch, heads, tokens, dtype=torch.float32)
        if op == "flash_train":
            state["dout"] = randn(batch, tokens, heads, dim, factor=1.0)
            state["workspace"] = ops.flash_backward_workspace(batch, tokens, heads, kv_heads, dim)
            state["grads"] = tuple(torch.empty_like(state[name]) for name in ("query", "key", "value"))
    elif op in ("prefill_forward", "prefill_train"):
        tokens = case["tokens"]
        state["scale"] = configs.c_float((NOPE + ROPE) ** -0.5)
        state["query"] = randn(batch, tokens, heads, NOPE + ROPE, factor=0.5)
        state["key"] = randn(batch, tokens, heads, NOPE + ROPE, factor=0.5)
        state["value"] = randn(batch, tokens, heads, VALUE, factor=0.5)
        for name in ("query", "key"):
            ops.rope_apply(state[name], rope_offset=NOPE)
        state["out"] = empty(batch, tokens, heads, VALUE)
        state["lse"] = empty(batch, heads, tokens, dtype=torch.float32)
        if op == "prefill_train":
            state["dout"] = randn(batch, tokens, heads, VALUE, factor=1.0)
            state["workspace"] = ops.mla_prefill_backward_workspace(batch, tokens, heads, NOPE + ROPE, VALUE)
            state["grads"] = tuple(torch.empty_like(state[name]) for name in ("query", "key", "value"))
    elif op in ("decode", "decode_layer"):
        lengths = _lengths(case)
        pages = [(length + PAGE - 1) // PAGE for length in lengths]
        # a pool of pages in the order a server hands them out: any page, to any sequence
        order = torch.randperm(sum(pages), device="cuda", generator=generator).to(torch.int32)
        table = torch.zeros(batch, max(pages), device="cuda", dtype=torch.int32)
        first = 0
        for row, count in enumerate(pages):
            table[row, :count] = order[first:first + count]
            first += count
        state["table"] = table
        state["cache"] = randn(sum(pages), PAGE, 1, RANK + ROPE, factor=0.5)
        state["lengths"] = torch.tensor(lengths, device="cuda", dtype=torch.int32)
        state["scale"] = configs.c_float((NOPE + ROPE) ** -0.5)
        state["workspace"] = ops.mla_decode_workspace(batch, heads, SPLITS)
        state["out"] = empty(batch, 1, heads, RANK)
        state["lse"] = empty(batch, heads, 1, dtype=torch.float32)
        if op == "decode":
            state["query"] = randn(batch, 1, heads, RANK + ROPE, factor=0.5)
        else:
            state["query_nope"] = randn(batch, 1, heads, NOPE, factor=0.5)
            state["query_rope"] = randn(batch, 1, heads, ROPE, factor=0.5)
            state["wkv_b"] = randn(heads, NOPE + VALUE, RANK, factor=0.06)
            state["query"] = empty(batch, 1, heads, RANK + ROPE)
            state["positions"] = state["lengths"] - 1
            state["plan"] = ops.mla_decode_plan(state["lengths"], heads, SPLITS)
            state["result"] = empty(batch, 1, heads, VALUE)
    else:
        tokens = case["tokens"]
        state["scale"] = configs.c_float((RANK + ROPE) ** -0.5)
        state["query_rope"] = randn(batch, tokens, heads, ROPE, factor=0.25)
        state["latent"] = randn(batch, tokens, RANK, factor=0.25)
        state["key_rope"] = randn(batch, tokens, ROPE, factor=0.25)
        state["query_latent"] = randn(batch, tokens, heads, RANK, factor=0.25)
        state["out"] = empty(batch, tokens, heads, RANK)
        state["lse"] = empty(batch, heads, tokens, dtype=torch.float32)
        if op == "absorbed_layer":
            state["query_nope"] = randn(batch, tokens, heads, NOPE, factor=0.5)
            state["wkv_b"] = randn(heads, NOPE + VALUE, RANK, factor=0.06)
            state["result"] = empty(batch, tokens, heads, VALUE)
        else:
            state["dout"] = randn(batch, tokens, heads, RANK, factor=0.2)
            state["grads"] = tuple(torch.empty_like(state[name])
                                   for name in ("query_latent", "query_rope", "latent", "key_rope"))
    return state


# ---- one pass ---------------------------------------------------------------------------------------------------

def run(state):
    op, scale = state["op"], state["scale"]
    if op in ("flash_forward", "flash_train"):
        operands = (state["query"], state["key"], state["value"])
        out, lse = ops.flash_forward(*operands, scale, state["out"], state["lse"])
        if op == "flash_forward":
            return out, lse
        grads = ops.flash_backward(state["dout"], out, lse, *operands, scale, state["workspace"], state["grads"])
        return (out, lse, *grads)
    if op in ("prefill_forward", "prefill_train"):
        operands = (state["query"], state["key"], state["value"])
        out, lse = ops.mla_prefill_forward(*operands, scale, state["out"], state["lse"])
        if op == "prefill_forward":
            return out, lse
        grads = ops.mla_prefill_backward(state["dout"], out, lse, *operands, scale, state["workspace"], state["grads"])
        return (out, lse, *grads)
    if op == "decode":
        return ops.mla_decode(state["query"], state["cache"], state["table"], state["lengths"], scale, splits=SPLITS,
                              workspace=state["workspace"], out=state["out"], lse=state["lse"])
    if op == "decode_layer":
        query, wkv_b = state["query"], state["wkv_b"]
        ops.mla_absorb_query(state["query_nope"], wkv_b[:, :NOPE], out=query[..., :RANK])
        query[..., RANK:].copy_(state["query_rope"])
        ops.rope_apply(query, rope_offset=RANK, positions=state["positions"])
        out, lse = ops.mla_decode_planned(query, state["cache"], state["table"], state["lengths"], state["plan"], scale,
                                          splits=SPLITS, workspace=state["workspace"], out=state["out"], lse=state["lse"])
        return ops.mla_unabsorb_output(out, wkv_b[:, NOPE:], out=state["result"]), out, lse, query
    operands = (state["query_latent"], state["query_rope"], state["latent"], state["key_rope"])
    if op == "absorbed_layer":
        ops.mla_absorb_query(state["query_nope"], state["wkv_b"][:, :NOPE], out=state["query_latent"])
        out, lse = ops.mla_forward(*operands, scale, state["out"], state["lse"])
        result = ops.mla_unabsorb_output(out, state["wkv_b"][:, NOPE:], out=state["result"])
        return result, out, lse, state["query_latent"]
    out, lse = ops.mla_forward(*operands, scale, state["out"], state["lse"])
    grads = ops.mla_backward(state["dout"], out, lse, *operands, scale, state["grads"])
    return (out, lse, *grads)


# ---- what one pass cannot do without ------------------------------------------------------------------------------

def _lengths(case):
    return configs.decode_lengths(case["batch"], case["low"], case["high"])[0].tolist()


def work(case):
    """Every input read once, every output written once (2 bytes an element, 4 of the logsumexp); the products over
    the T^2 / 2 visible pairs of a causal pass or over the cached tokens, five products for a backward."""
    op, batch, heads = case["op"], case["batch"], case["heads"]
    if op in ("flash_forward", "flash_train"):
        tokens, kv_heads, dim = case["tokens"], case["kv_heads"], case["dim"]
        rows, kv_rows = batch * tokens * heads, batch * tokens * kv_heads
        moved = 2 * dim * (2 * rows + 2 * kv_rows) + 4 * rows
        flops = configs.forward_flops(batch, heads, tokens, dim, dim)
        if op == "flash_train":
            moved += 2 * dim * (2 * rows + 2 * kv_rows)     # dO; dQ, dK, dV
            flops += configs.backward_flops(batch, heads, tokens, dim, dim)
    elif op in ("prefill_forward", "prefill_train"):
        tokens = case["tokens"]
        rows = batch * tokens * heads
        moved = rows * (2 * (2 * (NOPE + ROPE) + 2 * VALUE) + 4)
        flops = configs.forward_flops(batch, heads, tokens, NOPE + ROPE, VALUE)
        if op == "prefill_train":
            moved += rows * 2 * (2 * (NOPE + ROPE) + 2 * VALUE)
            flops += configs.backward_flops(batch, heads, tokens, NOPE + ROPE, VALUE)
    elif op in ("decode", "decode_layer"):
        total = sum(_lengths(case))
        flops = configs.decode_flops(total, heads)
        if op == "decode":
            moved = configs.decode_bytes(total, batch, heads)
        else:
            moved = (2 * total * (RANK + ROPE) + 2 * heads * (NOPE + VALUE) * RANK +
                     batch * heads * (2 * (NOPE + ROPE + VALUE) + 4))
            flops += 2 * batch * heads * (NOPE + VALUE) * RANK
    else:
        tokens = case["tokens"]
        rows, width = batch * tokens * heads, RANK + ROPE
        flops = batch * heads * (tokens * tokens / 2) * 2 * (width + RANK)
        if op == "absorbed_layer":
            moved = 2 * (rows * (NOPE + ROPE + VALUE) + batch * tokens * width + heads * (NOPE + VALUE) * RANK) + 4 * rows
            flops += 2 * rows * (NOPE + VALUE) * RANK
        else:
            moved = 2 * (rows * (width + RANK) + batch * tokens * width) + 4 * rows
            moved += 2 * (rows * (width + RANK) + batch * tokens * width)
            flops += batch * heads * (tokens * tokens / 2) * 2 * (3 * width + 2 * RANK)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """bf16 results with fp32 sums.  Against the same mathematics in fp64 the outputs of a forward differ by 1.9e-3 to
    2.8e-3 (their own rounding and that of the probabilities), gradients and what follows a projection by up to 3.3e-3
    (rounded once more on the way); four times that covers any other order of sums and roundings."""
    return {"rel": 8e-3 if case["op"] in ("flash_forward", "prefill_forward", "decode") else 1.2e-2}
