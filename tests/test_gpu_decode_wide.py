"""Absorbed decode with 128 heads a workgroup over pages that hold whole units of 32 keys (csrc/mla_wide.hip), and the plan
of a call at the batch sizes where its scan changes (64 sequences a wave, 256 a workgroup): sequences that end inside a unit,
a tile or a page, have one unit, are cut in the middle of a page, or are walked a second time."""

import pytest
import torch

from dscuda_amd.harness import configs, ops
from oracle import attention_oracle as oracle
from parity import announce, assert_close_bf16, assert_close_lse

pytestmark = pytest.mark.gpu

EDGES = [1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 191, 192, 193, 300, 511, 512, 513, 700]


def _inputs(batch, heads, page_size, lengths, seed):
    g = torch.Generator().manual_seed(seed)
    lengths = [lengths[i % len(lengths)] for i in range(batch)]
    query = (torch.randn(batch, 1, heads, 576, generator=g) * 0.25).bfloat16()
    cache = (torch.randn(batch, max(lengths), 576, generator=g) * 0.25).bfloat16()
    paged, table = configs.pack_cache(cache, page_size)
    order = torch.randperm(paged.shape[0], generator=g)
    inverse = torch.empty_like(order)
    inverse[order] = torch.arange(order.numel())
    return query, cache, paged[order].contiguous(), inverse[table.long()].to(torch.int32), torch.tensor(lengths, dtype=torch.int32)


@pytest.mark.parametrize("batch,heads,page_size,splits,lengths", [
    (25, 128, 64, 8, EDGES),
    (25, 128, 32, 8, EDGES),         # a page a unit
    (30, 97, 96, 8, EDGES),          # a last row block of one head; pages of three units, half of them cut by tiles
    (27, 257, 128, 8, EDGES[::-1]),  # three head groups, the last of one head
    (33, 128, 1024, 8, EDGES),       # one page a sequence
    (25, 128, 64, 1, EDGES),         # a workgroup a sequence
    (25, 100, 160, 2, EDGES),        # fewer slots than compute units
    (63, 128, 64, 8, [200, 33, 1, 90]), (64, 128, 64, 8, [200, 33, 1, 90]), (65, 128, 64, 8, [200, 33, 1, 90]),
    (257, 65, 64, 8, [70, 5, 40]),   # a plan by a kernel of its own
    (64, 16, 64, 8, [200, 33, 1, 90]), (65, 16, 64, 8, [200, 33, 1, 90]), (40, 64, 64, 8, EDGES), (1, 128, 64, 8, [700]),
    (64, 16, 48, 2, [13, 400]), (25, 128, 48, 8, EDGES),
    (255, 128, 48, 8, [70, 5, 40]), (256, 128, 48, 8, [70, 5, 40, 300]), (256, 128, 64, 8, [70, 5, 40, 300]),   # as many sequences as a
    (256, 16, 48, 8, [70, 5, 40, 300]), (257, 128, 48, 8, [70, 5, 40, 300]),                                    # workgroup plans for
])
def test_decode(cuda, batch, heads, page_size, splits, lengths):
    query, cache, paged, table, lengths_t = _inputs(batch, heads, page_size, lengths, seed=batch + heads)
    scale = configs.c_float(576 ** -0.5)
    announce("mla_decode", dict(B=batch, H=heads, page=page_size, splits=splits))
    # a table entry past the last page with a visible token is never used: such entries name a page of NaNs
    paged = torch.cat([paged, torch.full_like(paged[:1], float("nan"))])
    for row, length in enumerate(lengths_t.tolist()):
        table[row, (length + page_size - 1) // page_size:] = paged.shape[0] - 1
    on_gpu = [x.to(cuda) for x in (query, paged, table, lengths_t)]
    # an entry of the plan that the call does not write for itself stands for no sequence
    workspace = ops.mla_decode_workspace(batch, heads, splits).zero_()
    out, lse = ops.mla_decode(*on_gpu, scale, splits=splits, workspace=workspace)
    plan = ops.mla_decode_plan(on_gpu[3], heads, splits)
    planned, planned_lse = ops.mla_decode_planned(*on_gpu, plan, scale, splits=splits)
    torch.cuda.synchronize()
    expected, expected_lse = oracle.mla_decode_unrounded(query, cache, lengths_t, scale)
    assert_close_bf16("O", out, expected)
    assert_close_lse("LSE", lse, expected_lse)
    assert torch.equal(out, planned) and torch.equal(lse, planned_lse)


@pytest.mark.parametrize("splits,lengths,hot", [
    (1, [300, 40, 33], [(200, 260, 4.0), (36, 38, 4.0)]),
    (8, [1500, 1250, 64], [(600, 650, 1.0), (1000, 1100, 4.0)]),
])
def test_items_walked_again(cuda, splits, lengths, hot):
    """Scores that outgrow the first unit's by more than 2^80: the items of a workgroup that meet them are walked a second
    time, those around them once."""
    batch, heads = 26, 96
    g = torch.Generator().manual_seed(12)
    lengths = torch.tensor([lengths[i % len(lengths)] for i in range(batch)], dtype=torch.int32)
    query = torch.randn(batch, 1, heads, 576, generator=g).bfloat16()
    cache = (torch.randn(batch, int(lengths.max()), 576, generator=g) * 0.05).bfloat16()
    for first, last, factor in hot:
        cache[::2, first:last] = (query[::2, 0, :1].float() * factor).bfloat16()
    paged, table = configs.pack_cache(cache, 64)
    announce("mla_decode, items walked again", dict(splits=splits, hot=hot))
    out, lse = ops.mla_decode(query.to(cuda), paged.to(cuda), table.to(cuda), lengths.to(cuda), 1.0, splits=splits)
    expected, expected_lse = oracle.mla_decode_unrounded(query, cache, lengths, 1.0)
    assert expected_lse.max() > 500
    # outputs of these rows reach 15, where bf16 is spaced 0.06 apart, twice rounded where a sequence is cut
    torch.testing.assert_close(out.cpu().float(), expected, atol=8e-3, rtol=8e-3)
    assert ((lse.cpu() - expected_lse).abs() / expected_lse.abs().clamp_min(1)).max().item() <= 1e-5
