"""Absorbed prefill forward with 128 rows a workgroup (csrc/mla_wide.hip): a workgroup walks one item after the other, so
sizes at which items have one unit of keys or a few, end inside a unit or a row block, change the batch element, or are
walked a second time; both sides of the rule that sends a call there."""

import pytest
import torch

from dscuda_amd.harness import configs, ops
from dispatch_rules import rules
from oracle import attention_oracle as oracle
from parity import announce, assert_close_bf16, assert_close_lse

pytestmark = pytest.mark.gpu


# 171 and 256 workgroups of 128 rows are two thirds and the whole of one round, 320 one and a quarter
@pytest.mark.parametrize("batch,tokens,heads,rows", [
    (1, 171, 128, 64), (1, 170, 128, 64), (1, 256, 128, 64), (2, 383, 42, 64), (2, 385, 42, 64), (1, 257, 128, 128),
    (1, 160, 139, 128), (1, 161, 139, 64), (1, 224, 146, 128), (4, 383, 21, 128), (3, 225, 32, 64), (3, 256, 34, 128),
    (1, 672, 49, 128), (1, 673, 49, 64),   # 258 workgroups, walks of 21 and 22 units
    (321, 5, 25, 128), (320, 5, 25, 64), (320, 33, 3, 128), (257, 1, 129, 128),
    (3, 97, 129, 128),    # a row block over two tokens, items of two, three and four units
    (7, 161, 40, 128),    # batch elements end inside a row block and a unit; two rounds
    (70, 40, 64, 128),    # 1400 items of two units
    (1, 515, 131, 128),   # three rounds, the last of 16 items
    (2, 1500, 30, 128),   # keys of both elements together do not fit an L2; their blocks are numbered together all the same
    (4, 1024, 32, 128),   # such keys, and elements that fill rounds: one element after the other
])
def test_forward(cuda, batch, tokens, heads, rows):
    units = torch.cuda.get_device_properties(cuda).multi_processor_count
    if units == 256:
        assert rules().forward_rows(batch, tokens, heads, units) == rows
    ql, qr, c, kr, scale = configs.mla_absorbed_inputs(batch, tokens, heads)
    announce("mla_forward, 128 rows", dict(B=batch, T=tokens, H=heads))
    on_gpu = [x.to(cuda) for x in (ql, qr, c, kr)]
    out, lse = ops.mla_forward(*on_gpu, scale, out=torch.full_like(on_gpu[0], float("nan")))
    again, lse_again = ops.mla_forward(*on_gpu, scale)
    assert torch.equal(out, again) and torch.equal(lse, lse_again)
    # the first, the last and some elements between against the oracle (the references of all 321 would take minutes)
    some = sorted({0, 1, batch // 2, batch - 1} & set(range(batch)))
    expected, expected_lse = oracle.mla_forward_unrounded(ql[some], qr[some], c[some], kr[some], scale, oracle.causal_mask(tokens))
    assert_close_bf16("O", out[some], expected, max_abs=8e-3)
    assert_close_lse("LSE", lse[some], expected_lse, tol=1e-4)
    assert torch.isfinite(out).all() and torch.isfinite(lse).all()


def test_items_walked_again(cuda):
    """Scores beyond 2^80 times the first unit's in some rows of some items, the first and the last of a workgroup's among
    them: those items are walked a second time, the ones after them go on as before.  Weights carry the fp32 error of
    scores of this size (see test_gpu_row_blocks.assert_rounded)."""
    tokens, heads = 400, 300
    g = torch.Generator().manual_seed(3)
    ql, qr, c, kr, _ = configs.mla_absorbed_inputs(1, tokens, heads)
    for token, head in [(50, 0), (51, 299), (200, 7), (399, 150)]:
        ql[0, token, head] = torch.randn(512, generator=g).bfloat16()
        c[0, token - 12] = ql[0, token, head]
    announce("mla_forward, items walked again", dict(T=tokens, H=heads))
    out, lse = ops.mla_forward(*(x.to(cuda) for x in (ql, qr, c, kr)), 1.0)
    expected, expected_lse = oracle.mla_forward_unrounded(ql, qr, c, kr, 1.0, oracle.causal_mask(tokens))
    assert expected_lse.max() > 400
    weights = 40 * 2 ** -24 * expected_lse.abs().max().item()
    error = (out.cpu().float() - expected).abs()
    assert error.max().item() <= (3 * 2 ** -9 + weights) * c.float().abs().max().item() and error.mean().item() <= 6e-3
    assert ((lse.cpu() - expected_lse).abs() / expected_lse.abs().clamp_min(1)).max().item() <= 1e-5


def test_scores_too_large_for_their_own_rounding(cuda):
    """Scores of 1e30 in some rows of some items: their distance from their rounded maximum is beyond any limit, a second walk
    is the last all the same.  What comes out for these rows is not asserted; all other rows, of the items walked twice and of
    those before and after them, are as ever, and every row is written."""
    tokens, heads = 400, 300
    ql, qr, c, kr, scale = configs.mla_absorbed_inputs(1, tokens, heads)
    huge = [(30, 0), (31, 299), (200, 7), (200, 130), (399, 150)]
    for token, head in huge:
        ql[0, token, head] *= 1e30
    announce("mla_forward, huge scores", dict(T=tokens, H=heads))
    on_gpu = [x.to(cuda) for x in (ql, qr, c, kr)]
    untouched = -77.0
    runs = []
    for _ in range(2):
        out, lse = torch.full_like(on_gpu[0], untouched), torch.full((1, heads, tokens), untouched, device=cuda)
        ops.mla_forward(*on_gpu, scale, out=out, lse=lse)
        runs.append((out.view(torch.int16), lse.view(torch.int32)))
    torch.cuda.synchronize()
    assert torch.equal(runs[0][0], runs[1][0]) and torch.equal(runs[0][1], runs[1][1])
    assert not (out == untouched).all(-1).any() and not (lse == untouched).any()
    ordinary = torch.ones(1, tokens, heads, dtype=torch.bool)
    for token, head in huge:
        ordinary[0, token, head] = False
        ql[0, token, head] = 0
    expected, expected_lse = oracle.mla_forward_unrounded(ql, qr, c, kr, scale, oracle.causal_mask(tokens))
    assert_close_bf16("O", out.cpu()[ordinary], expected[ordinary], max_abs=8e-3)
    assert_close_lse("LSE", lse.cpu().transpose(1, 2)[ordinary], expected_lse.transpose(1, 2)[ordinary], tol=1e-4)
