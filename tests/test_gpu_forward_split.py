"""The split-key and the persistent forward at the edges of their tiles (32, 64 and 128 queries or keys), of their work
order (head counts that are dealt to the XCDs by group, by head or not at all) and of the line between them."""

import pytest
import torch

from dscuda_amd.harness import configs, ops
from oracle import attention_oracle as oracle
from tests.parity import announce, assert_close_bf16, assert_close_lse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,seq,heads", [
    (1, 31, 1), (1, 32, 2), (3, 33, 1), (1, 63, 3), (1, 64, 8), (2, 65, 4), (1, 127, 5), (1, 128, 16), (1, 129, 3),
    (1, 191, 2), (2, 193, 8), (1, 256, 3), (1, 320, 1),                      # 64 queries per workgroup
    (1, 130, 70), (2, 129, 68), (1, 385, 40), (1, 257, 96),                  # 128
    (1, 1024, 128), (1, 640, 160),                                           # persistent
])
def test_prefill_tile_edges(cuda, batch, seq, heads):
    q, k, v, scale = configs.mla_prefill_inputs(batch, seq, heads, seed=seq)
    announce("prefill tile edges", dict(B=batch, S=seq, H=heads))
    out, lse = ops.mla_prefill_forward(q.to(cuda), k.to(cuda), v.to(cuda), scale)
    sample = sorted({0, heads // 2, heads - 1})
    expected, expected_lse = oracle.causal_attention_forward(q, k, v, scale, heads=sample)
    assert_close_bf16("O", out[:, :, sample], expected)
    assert_close_lse("LSE", lse[:, sample], expected_lse)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("batch,tokens,kv_heads,sharing", [
    (1, 192, 8, 3), (2, 64, 4, 1), (1, 128, 1, 8), (3, 320, 1, 5), (1, 448, 24, 4),
])
def test_flash_work_orders(cuda, batch, tokens, kv_heads, sharing, dim):
    heads = kv_heads * sharing
    q, k, v, scale = configs.flash_forward_inputs(batch, tokens, heads, kv_heads, dim, seed=tokens, factor=0.5)
    announce("flash work orders", dict(B=batch, T=tokens, Hq=heads, Hkv=kv_heads, D=dim))
    out, lse = ops.flash_forward(q.to(cuda), k.to(cuda), v.to(cuda), scale)
    expected, expected_lse = oracle.causal_attention_forward(q, k, v, scale)
    assert_close_bf16("O", out, expected)
    assert_close_lse("LSE", lse, expected_lse)


@pytest.mark.parametrize("batch,tokens,heads,kv_heads", [
    (3, 64, 128, 128), (4, 192, 96, 32), (24, 128, 16, 16), (2, 192, 128, 16), (1, 320, 224, 56), (1, 384, 256, 64),
    (1, 448, 384, 48), (1, 2112, 256, 2),   # four waves
    (2, 448, 128, 32), (1, 128, 256, 64), (1, 192, 223, 223), (1, 64, 127, 127),   # the other side of the rule
    (1, 1280, 67, 67), (3, 896, 33, 11), (1, 576, 155, 31),   # heads dealt to the XCDs with slots left over
])
def test_flash_64_columns_many_heads(cuda, batch, tokens, heads, kv_heads):
    q, k, v, scale = configs.flash_forward_inputs(batch, tokens, heads, kv_heads, 64, seed=tokens, factor=0.5)
    announce("flash, many heads", dict(B=batch, T=tokens, Hq=heads, Hkv=kv_heads))
    out, lse = ops.flash_forward(q.to(cuda), k.to(cuda), v.to(cuda), scale)
    sample = sorted({0, heads // 2, heads - 1})
    group = heads // kv_heads
    own = [h // group for h in sample]
    expected, expected_lse = oracle.causal_attention_forward(q[:, :, sample], k[:, :, own], v[:, :, own], scale)
    assert_close_bf16("O", out[:, :, sample], expected)
    assert_close_lse("LSE", lse[:, sample], expected_lse)


@pytest.mark.parametrize("dqk", [192, 128])
@pytest.mark.parametrize("batch,seq,heads", [(1, 1, 128), (3, 31, 130), (2, 33, 64), (9, 64, 16), (2, 65, 64), (1, 64, 127)])
def test_one_tile_of_keys(cuda, batch, seq, heads, dqk):
    g = torch.Generator().manual_seed(seq)
    randn = lambda dim: (torch.randn(batch, seq, heads, dim, generator=g) * 0.5).bfloat16()
    q, k, v = randn(dqk), randn(dqk), randn(128)
    scale = configs.c_float(dqk ** -0.5)
    announce("one tile of keys", dict(B=batch, S=seq, H=heads, dqk=dqk))
    out, lse = ops.mla_prefill_forward(q.to(cuda), k.to(cuda), v.to(cuda), scale)
    expected, expected_lse = oracle.causal_attention_forward(q, k, v, scale)
    assert_close_bf16("O", out, expected)
    assert_close_lse("LSE", lse, expected_lse)


@pytest.mark.parametrize("heads", [2, 72])   # 64 and 128 queries per workgroup
def test_parts_with_distant_maxima(cuda, heads):
    """Scores that grow by thousands along the keys: the key groups of a workgroup end with maxima far apart, and rows
    near a tile's start have no visible key in some of them."""
    seq = 300
    g = torch.Generator().manual_seed(3)
    direction = torch.randn(192, generator=g)
    q = (direction + 0.1 * torch.randn(1, seq, heads, 192, generator=g)).bfloat16()
    growth = torch.linspace(0, 1, seq)[None, :, None, None]
    k = (direction * growth + 0.05 * torch.randn(1, seq, heads, 192, generator=g)).bfloat16()
    v = torch.randn(1, seq, heads, 128, generator=g).bfloat16()
    announce("distant maxima", dict(H=heads))
    out, lse = ops.mla_prefill_forward(q.to(cuda), k.to(cuda), v.to(cuda), 4.0)
    expected, expected_lse = oracle.causal_attention_forward(q, k, v, 4.0)
    assert expected_lse.max() > 500
    # the weights carry the fp32 error of scores this large: twelve partial sums and the scaling, 2^-24 of the score each
    weights = 16 * 2 ** -24 * expected_lse.abs().max().item()
    largest = v.float().abs().max().item()
    assert (out.cpu().float() - expected).abs().max().item() <= (2 * 2 ** -9 + weights) * largest
    assert ((lse.cpu() - expected_lse).abs() / expected_lse.abs().clamp_min(1)).max().item() <= 1e-5


@pytest.mark.parametrize("heads", [2, 72])   # 64 and 128 queries per workgroup
def test_scores_far_below_zero_under_a_small_scale(cuda, heads):
    """Raw scores of -4e33 under a scale that brings them to some -400: the running maximum has to start below every
    score, and key groups that a row's queries never reach must not count."""
    seq = 200
    g = torch.Generator().manual_seed(4)
    randn = lambda dim: torch.randn(1, seq, heads, dim, generator=g)
    q = (2.0 ** 52 * (1 + 0.05 * randn(192))).bfloat16()
    k = (-2.0 ** 52 * (1 + 0.05 * randn(192))).bfloat16()
    v = randn(128).bfloat16()
    scale = configs.c_float(1e-31)
    announce("scores far below zero", dict(H=heads))
    out, lse = ops.mla_prefill_forward(q.to(cuda), k.to(cuda), v.to(cuda), scale)
    expected, expected_lse = oracle.causal_attention_forward(q, k, v, scale)
    assert expected_lse.max() < -300
    # the weights carry the fp32 error of the scores: twelve partial sums and the scaling, 2^-24 of the score each
    weights = 16 * 2 ** -24 * expected_lse.abs().max().item()
    largest = v.float().abs().max().item()
    assert (out.cpu().float() - expected).abs().max().item() <= (2 * 2 ** -9 + weights) * largest
    assert ((lse.cpu() - expected_lse).abs() / expected_lse.abs()).max().item() <= 1e-5


@pytest.mark.parametrize("seq,heads,dim", [(64, 600000, 64), (128, 140000, 128), (192, 280000, 128)])
def test_query_rows_four_gigabytes_apart(cuda, seq, heads, dim):
    """One key/value head for so many query heads that the last query row of a tile (64 rows, 128, and a last one of 64)
    lies more than 4 GiB behind its first."""
    rows = 128 if seq == 128 else 64
    assert (rows - 1) * heads * dim * 2 > 2 ** 32
    g = torch.Generator(device=cuda).manual_seed(5)
    q = torch.empty(1, seq, heads, dim, device=cuda, dtype=torch.bfloat16).normal_(0, 0.5, generator=g)
    k, v = (torch.empty(1, seq, 1, dim, device=cuda, dtype=torch.bfloat16).normal_(0, 0.5, generator=g) for _ in range(2))
    scale = configs.c_float(dim ** -0.5)
    announce("query rows far apart", dict(S=seq, Hq=heads, D=dim))
    out, lse = ops.flash_forward(q, k, v, scale)
    sample = [0, heads // 2, heads - 1]
    expected, expected_lse = oracle.causal_attention_forward(q[:, :, sample].cpu(), k.cpu(), v.cpu(), scale)
    assert_close_bf16("O", out[:, :, sample], expected)
    assert_close_lse("LSE", lse[:, sample], expected_lse)
