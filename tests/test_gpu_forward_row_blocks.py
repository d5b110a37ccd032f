"""Absorbed forward where 32-row workgroups would take a second round: sizes on both sides of the choice between 32 and 64
rows, rows that end inside a workgroup, several batch elements, more heads than a workgroup has rows."""

import pytest
import torch

from dscuda_amd.harness import configs, ops
from dispatch_rules import rules
from oracle import attention_oracle as oracle
from parity import announce, assert_close_bf16, assert_close_lse

pytestmark = pytest.mark.gpu


# 64 x 128 rows are one round of 32-row workgroups, one token more two; 433 and 434 tokens of 32 heads, 140 and 141 of 64 the
# two sides of the sums; 300 x 1 x 40 and the last three are chosen by the number of 128-row workgroups
@pytest.mark.parametrize("batch,tokens,heads,rows", [
    (1, 65, 127, 64), (1, 100, 128, 64), (1, 127, 128, 64), (3, 299, 16, 64), (8, 250, 8, 64), (1, 250, 64, 64), (1, 400, 32, 32),
    (300, 1, 40, 64), (16, 33, 31, 64), (1, 64, 128, 32), (1, 65, 128, 64), (1, 433, 32, 32),
    (1, 434, 32, 64), (1, 140, 64, 32), (1, 141, 64, 64), (1, 129, 128, 64), (320, 3, 42, 64), (321, 3, 42, 128)])
def test_forward(cuda, batch, tokens, heads, rows):
    units = torch.cuda.get_device_properties(cuda).multi_processor_count
    if units == 256:
        assert rules().forward_rows(batch, tokens, heads, units) == rows
    ql, qr, c, kr, scale = configs.mla_absorbed_inputs(batch, tokens, heads)
    announce("mla_forward, 32 or 64 rows", dict(B=batch, T=tokens, H=heads))
    out, lse = ops.mla_forward(*(x.to(cuda) for x in (ql, qr, c, kr)), scale)
    torch.cuda.synchronize()
    expected, expected_lse = oracle.mla_forward_unrounded(ql, qr, c, kr, scale, oracle.causal_mask(tokens))
    assert_close_bf16("O", out, expected, max_abs=8e-3)
    assert_close_lse("LSE", lse, expected_lse, tol=1e-4)
