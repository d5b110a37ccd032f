"""The three forms of the absorbed decode and prefill forward (32, 64 and 128 rows per workgroup) at the edges of
their row groups, key units and dispatch ranges, against the fp32 oracle; and the raised softmax reference in each."""

import pytest
import torch

from dscuda_amd.harness import configs, ops
from oracle import attention_oracle as oracle
from tests.dispatch_rules import rules
from tests.parity import announce, assert_close_bf16, assert_close_lse

pytestmark = pytest.mark.gpu


def assert_rounded(out, expected, expected_lse, values):
    """Probabilities, partial rows and results are each rounded to bf16 once, by at most 2^-9 of a mean of |values|
    that the softmax weights; the weights themselves carry the fp32 error of scores this large: 36 partial sums, the
    scaling and the two log-sum-exp steps round by 2^-24 of the score each."""
    largest = values.float().abs().max().item()
    weights = 40 * 2 ** -24 * expected_lse.abs().max().item()
    error = (out.cpu().float() - expected).abs()
    worst, mean = error.max().item(), error.mean().item()
    assert worst <= (3 * 2 ** -9 + weights) * largest and mean <= 6e-3


@pytest.mark.parametrize("batch,heads,splits", [
    (7, 1, 8), (7, 15, 8), (7, 17, 4), (7, 32, 8), (7, 32, 1),   # 32 rows, one head group
    (7, 33, 8), (2, 65, 8), (7, 128, 1),                          # 32 rows, every range has its compute units
    (14, 64, 8), (14, 47, 8), (14, 65, 8), (14, 100, 3),          # 64 rows
    (28, 128, 8), (28, 97, 2),                                    # 128 rows
])
def test_decode_row_blocks(cuda, batch, heads, splits):
    lengths = ([1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 129, 200, 700] * 2)[:batch]
    tokens = max(lengths)
    g = torch.Generator().manual_seed(batch + heads)
    query = (torch.randn(batch, 1, heads, 576, generator=g) * 0.25).bfloat16()
    cache = (torch.randn(batch, tokens, 576, generator=g) * 0.25).bfloat16()
    paged, table = configs.pack_cache(cache, 64)
    lengths = torch.tensor(lengths, dtype=torch.int32)
    scale = configs.c_float(576 ** -0.5)
    announce("decode row blocks", dict(B=batch, H=heads, splits=splits))
    out, lse = ops.mla_decode(query.to(cuda), paged.to(cuda), table.to(cuda), lengths.to(cuda), scale, splits=splits)
    expected, expected_lse = oracle.mla_decode_unrounded(query, cache, lengths, scale)
    assert_close_bf16("O", out, expected)
    assert_close_lse("LSE", lse, expected_lse)


# 32, 64 and 128 rows; 128 rows over pages that hold no whole units of 32 keys, which have a kernel of their own
@pytest.mark.parametrize("batch,heads,page_size,rows", [(2, 40, 64, 32), (14, 64, 64, 32), (24, 128, 64, 64),
                                                        (28, 128, 64, 128), (28, 128, 48, 128), (28, 97, 16, 128)])
def test_decode_raised_reference(cuda, batch, heads, page_size, rows):
    """Keys late in the stream aligned with one head of each row group: scores thousands above the first keys'."""
    units = torch.cuda.get_device_properties(cuda).multi_processor_count
    assert {0: 128, 1: 32, 2: 64}[rules().call_rows(batch, heads, 2, page_size, units)] == rows
    tokens = 420
    g = torch.Generator().manual_seed(31)
    query = torch.randn(batch, 1, heads, 576, generator=g).bfloat16()
    cache = (torch.randn(batch, tokens, 576, generator=g) * 0.05).bfloat16()
    for first, last, head, factor in [(70, 72, 0, 1.0), (200, 201, heads - 1, 2.0), (300, 340, heads // 2, 4.0)]:
        cache[:, first:last] = (query[:, 0, head:head + 1].float() * factor).bfloat16()
    lengths = torch.tensor([tokens - 11 * (b % 9) for b in range(batch)], dtype=torch.int32)
    paged, table = configs.pack_cache(cache, page_size)
    announce("decode raised reference", dict(B=batch, H=heads, page=page_size))
    out, lse = ops.mla_decode(query.to(cuda), paged.to(cuda), table.to(cuda), lengths.to(cuda), 1.0, splits=2)
    expected, expected_lse = oracle.mla_decode_unrounded(query, cache, lengths, 1.0)
    assert expected_lse.max() > 500
    assert_rounded(out, expected, expected_lse, cache)
    assert ((lse.cpu() - expected_lse).abs() / expected_lse.abs().clamp_min(1)).max().item() <= 1e-5


@pytest.mark.parametrize("batch,tokens,heads", [
    (1, 32, 1), (1, 33, 1), (3, 63, 2), (1, 129, 31),   # 32 rows, last block of 1, 2, 30 and 31 rows among them
    (1, 273, 63), (2, 129, 65), (1, 160, 127),          # 64 rows
    (1, 345, 120),                                      # 128 rows
])
def test_forward_row_blocks(cuda, batch, tokens, heads):
    ql, qr, c, kr, scale = configs.mla_absorbed_inputs(batch, tokens, heads, seed=tokens)
    announce("forward row blocks", dict(B=batch, T=tokens, H=heads))
    out, lse = ops.mla_forward(ql.to(cuda), qr.to(cuda), c.to(cuda), kr.to(cuda), scale)
    expected, expected_lse = oracle.mla_forward_unrounded(ql, qr, c, kr, scale, oracle.causal_mask(tokens))
    assert_close_bf16("O", out, expected, max_abs=8e-3)
    assert_close_lse("LSE", lse, expected_lse, tol=1e-4)


@pytest.mark.parametrize("tokens,heads", [(150, 64), (330, 128)])   # 64 and 128 rows
def test_forward_raised_reference(cuda, tokens, heads):
    g = torch.Generator().manual_seed(14)
    direction = torch.randn(576, generator=g)
    query = (direction[None, None, None, :] + 0.1 * torch.randn(1, tokens, heads, 576, generator=g)).bfloat16()
    keys = (torch.randn(1, tokens, 576, generator=g) * 0.05).bfloat16()
    for first, last, factor in [(50, 60, 1.0), (100, 130, 4.0)]:
        keys[:, first:last] = (direction * factor).bfloat16()
    ql, qr = query[..., :512].contiguous(), query[..., 512:].contiguous()
    c, kr = keys[..., :512].contiguous(), keys[..., 512:].contiguous()
    announce("forward raised reference", dict(T=tokens, H=heads))
    out, lse = ops.mla_forward(ql.to(cuda), qr.to(cuda), c.to(cuda), kr.to(cuda), 1.0)
    expected, expected_lse = oracle.mla_forward_unrounded(ql, qr, c, kr, 1.0, oracle.causal_mask(tokens))
    assert expected_lse.max() > 500
    assert_rounded(out, expected, expected_lse, c)
    assert ((lse.cpu() - expected_lse).abs() / expected_lse.abs().clamp_min(1)).max().item() <= 1e-5


@pytest.mark.parametrize("parts", [2, 15, 16, 17, 32, 33, 63, 64, 65, 81, 128])
def test_decode_merge_of_many_parts(cuda, parts):
    """One sequence cut into as many parts as it has tiles: rows are merged 16 parts, statistics 64 parts at a time."""
    heads, tokens = 3, 64 * parts - 5
    g = torch.Generator().manual_seed(parts)
    query = (torch.randn(1, 1, heads, 576, generator=g) * 0.25).bfloat16()
    cache = (torch.randn(1, tokens, 576, generator=g) * 0.25).bfloat16()
    paged, table = configs.pack_cache(cache, 64)
    lengths = torch.tensor([tokens], dtype=torch.int32)
    scale = configs.c_float(576 ** -0.5)
    announce("decode, merge of many parts", dict(T=tokens, H=heads))
    out, lse = ops.mla_decode(query.to(cuda), paged.to(cuda), table.to(cuda), lengths.to(cuda), scale, splits=128)
    expected, expected_lse = oracle.mla_decode_unrounded(query, cache, lengths, scale)
    assert_close_bf16("O", out, expected)
    assert_close_lse("LSE", lse, expected_lse)


@pytest.mark.parametrize("batch,heads,splits,low,high", [
    (1, 8, 8, 400, 400), (5, 8, 8, 33, 271), (3, 40, 8, 60, 300),   # more ranges than padded slots would allow
    (8, 16, 2, 300, 2000), (2, 24, 2, 300, 300),
    (300, 4, 2, 64, 200),                                            # the plan kernel
])
def test_sequences_that_fewer_ranges_leave_whole_are_rounded_once(cuda, batch, heads, splits, low, high):
    """Probabilities and results are rounded to bf16, parts of these sequences are not.  A rounding errs evenly within
    half a step of 2^-7 of the power of two below a value: 2^-7 / sqrt(12) over a root mean square of 1.36 (such powers)
    is 1.66e-3 in the 2-norm.  Two independent ones make 2.35e-3, a third one, of the parts, 2.88e-3."""
    g = torch.Generator().manual_seed(batch + heads)
    lengths = torch.linspace(low, high, batch).int()
    tokens = int(lengths.max())
    query = (torch.randn(batch, 1, heads, 576, generator=g) * 0.5).bfloat16()
    cache = (torch.randn(batch, tokens, 576, generator=g) * 0.5).bfloat16()
    paged, table = configs.pack_cache(cache, 64)
    scale = configs.c_float(192 ** -0.5)
    announce("decode, parts in fp32", dict(B=batch, H=heads, splits=splits, lengths=(low, high)))
    on_gpu = [x.to(cuda) for x in (query, paged, table, lengths)]
    out, lse = ops.mla_decode(*on_gpu, scale, splits=splits)
    plan = ops.mla_decode_plan(on_gpu[3], heads, splits)
    planned, planned_lse = ops.mla_decode_planned(*on_gpu, plan, scale, splits=splits)
    assert torch.equal(out, planned) and torch.equal(lse, planned_lse)
    expected, expected_lse = oracle.mla_decode_unrounded(query.double(), cache.double(), lengths, scale)
    error = (out.cpu().double() - expected).norm() / expected.norm()
    assert error.item() <= 2.6e-3
    assert_close_lse("LSE", lse, expected_lse)


@pytest.mark.parametrize("batch,heads,splits,page,high", [
    (20, 128, 8, 16, 600), (16, 96, 32, 1, 300), (17, 65, 8, 48, 2000),
])
def test_decode_pages_that_hold_no_whole_units(cuda, batch, heads, splits, page, high):
    """Calls whose plan is made for 64 rows but whose pages are looked up key by key run 128 rows over the plan's
    positions: the same ranges, and so the same bits, as without a plan."""
    units = torch.cuda.get_device_properties(cuda).multi_processor_count
    assert rules().plan_rows(batch, heads, splits, units) == 2 and rules().call_rows(batch, heads, splits, page, units) == 0
    g = torch.Generator().manual_seed(batch)
    lengths = torch.linspace(1, high, batch).int()
    query = (torch.randn(batch, 1, heads, 576, generator=g) * 0.25).bfloat16()
    cache = (torch.randn(batch, high, 576, generator=g) * 0.25).bfloat16()
    paged, table = configs.pack_cache(cache, page)
    scale = configs.c_float(576 ** -0.5)
    announce("decode, pages looked up", dict(B=batch, H=heads, splits=splits, page=page))
    on_gpu = [x.to(cuda) for x in (query, paged, table, lengths)]
    expected, expected_lse = oracle.mla_decode_unrounded(query, cache, lengths, scale)
    out, lse = ops.mla_decode(*on_gpu, scale, splits=splits)
    assert_close_bf16("O", out, expected)
    assert_close_lse("LSE", lse, expected_lse)
    plan = ops.mla_decode_plan(on_gpu[3], heads, splits)
    planned, planned_lse = ops.mla_decode_planned(*on_gpu, plan, scale, splits=splits)
    assert torch.equal(out, planned) and torch.equal(lse, planned_lse)


@pytest.mark.parametrize("batch,heads,splits,page,high", [
    (28, 128, 8, 64, 400), (70, 128, 1, 64, 200),      # parts, and a workgroup per sequence
    (260, 128, 8, 64, 130), (260, 128, 1, 64, 90),     # the plan kernel
    (28, 128, 8, 16, 300), (28, 128, 8, 48, 300),      # pages looked up key by key
    (28, 128, 8, 32, 2500),                            # page ids of two loads
    (25, 160, 8, 64, 300), (40, 200, 1, 16, 150),      # a second head group
])
def test_decode_of_128_rows(cuda, batch, heads, splits, page, high):
    """The 128-row form with its own plan and with the caller's, whose ranges are the same.  One sequence is empty: it
    owns no key and no result."""
    units = torch.cuda.get_device_properties(cuda).multi_processor_count
    assert rules().plan_rows(batch, heads, splits, units) == 0 and rules().call_rows(batch, heads, splits, page, units) == 0
    g = torch.Generator().manual_seed(batch + heads + page)
    lengths = torch.linspace(1, high, batch).int()
    lengths[batch // 3] = 0
    query = (torch.randn(batch, 1, heads, 576, generator=g) * 0.25).bfloat16()
    cache = (torch.randn(batch, high, 576, generator=g) * 0.25).bfloat16()
    paged, table = configs.pack_cache(cache, page)
    scale = configs.c_float(576 ** -0.5)
    announce("decode of 128 rows", dict(B=batch, H=heads, splits=splits, page=page, tokens=high))
    on_gpu = [x.to(cuda) for x in (query, paged, table, lengths)]
    out, lse = ops.mla_decode(*on_gpu, scale, splits=splits)
    plan = ops.mla_decode_plan(on_gpu[3], heads, splits)
    planned, planned_lse = ops.mla_decode_planned(*on_gpu, plan, scale, splits=splits)
    some = (lengths > 0).nonzero().flatten()
    expected, expected_lse = oracle.mla_decode_unrounded(query[some], cache[some], lengths[some], scale)
    assert_close_bf16("O", out.cpu()[some], expected)
    assert_close_lse("LSE", lse.cpu()[some], expected_lse)
    assert torch.equal(out.cpu()[some], planned.cpu()[some]) and torch.equal(lse.cpu()[some], planned_lse.cpu()[some])
