"""Absorbed forward where 32-row workgroups would take a second round: sizes on both sides of the choice between 32 and 64
rows, rows that end inside a workgroup, several batch elements, more heads than a workgroup has rows."""

import pytest
import torch

from dscuda_amd.harness import configs, ops
from oracle import attention_oracle as oracle
from parity import announce, assert_close_bf16, assert_close_lse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,tokens,heads", [
    (1, 65, 127), (1, 100, 128), (1, 127, 128), (3, 299, 16), (8, 250, 8), (1, 250, 64), (1, 400, 32), (300, 1, 40), (16, 33, 31)])
def test_forward(cuda, batch, tokens, heads):
    ql, qr, c, kr, scale = configs.mla_absorbed_inputs(batch, tokens, heads)
    announce("mla_forward, 32 or 64 rows", dict(B=batch, T=tokens, H=heads))
    out, lse = ops.mla_forward(*(x.to(cuda) for x in (ql, qr, c, kr)), scale)
    torch.cuda.synchronize()
    expected, expected_lse = oracle.mla_forward_unrounded(ql, qr, c, kr, scale, oracle.causal_mask(tokens))
    assert_close_bf16("O", out, expected, max_abs=8e-3)
    assert_close_lse("LSE", lse, expected_lse, tol=1e-4)
