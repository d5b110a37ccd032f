"""GPU parity of the absorbed backward of short sequences, which keeps P and dS in the query-gradient buffers
(index_math::short_backward; the placement itself is enumerated in tests/host/index_math_test.cpp), and of the same calls
with the workspace that the library asks for, which takes some of them to other kernels."""

import pytest
import torch

from dscuda_amd.harness import configs, ops
from oracle import attention_oracle as oracle
from tests.dispatch_rules import rules
from tests.parity import announce, assert_close_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,tokens,heads", [
    (1, 1, 1), (1, 32, 1), (1, 33, 1), (2, 31, 3),
    (1, 64, 2), (3, 65, 1),
    (1, 129, 5),       # a second key group of one key, row tiles that start inside tokens
    (1, 480, 3),       # fifteen whole blocks of tokens
    (1, 481, 3),       # a sixteenth of one token, whose P lies in the rope gradients
    (2, 511, 2),
    (1, 512, 8),       # the most tokens
    (1, 187, 32),      # 5984 rows, the most heads
    (7, 512, 4),       # 14336 rows over the batch
    (1, 513, 4), (1, 188, 32), (1, 100, 33),   # the other side of the rule
])
def test_absorbed_backward_of_short_sequences(cuda, batch, tokens, heads):
    ql, qr, c, kr, scale = configs.mla_absorbed_inputs(batch, tokens, heads)
    g = torch.Generator().manual_seed(91)
    dout = (torch.randn(batch, tokens, heads, 512, generator=g) * 0.2).bfloat16()
    mask = oracle.causal_mask(tokens)
    out, lse = oracle.mla_forward(ql, qr, c, kr, scale, mask)
    announce("mla_backward, short", dict(B=batch, T=tokens, H=heads))
    operands = tuple(x.to(cuda) for x in (dout, out, lse, ql, qr, c, kr))
    expected = oracle.mla_backward_unrounded(dout, out, lse, ql, qr, c, kr, scale, mask)
    for workspace in (torch.empty(0, device=cuda), None):   # dscuda_mla_backward, and the workspace the library asks for
        runs = []
        for _ in range(2):
            grads = tuple(torch.full_like(x, float("nan")) for x in operands[3:])   # scratch as well as results
            runs.append(ops.mla_backward(*operands, scale, grads, workspace))
        torch.cuda.synchronize()
        for name, first, second, reference in zip(("dq_latent", "dq_rope", "dlatent", "dk_rope"), *runs, expected):
            assert torch.equal(first, second)
            assert_close_bf16(name, first.cpu(), reference)


@pytest.mark.parametrize("batch,tokens,heads,kept", [
    (1, 33, 1, True), (1, 3, 11, True), (2, 2, 17, True), (9, 384, 1, True), (2, 219, 20, True),
    (12, 2, 17, True), (32, 16, 4, True), (16, 100, 1, True), (13, 2, 17, False), (33, 16, 4, False), (17, 100, 1, False),
    (1, 1, 32, False), (13, 4, 8, False), (10, 353, 2, False), (2, 224, 20, False), (2, 160, 32, False),
])
def test_which_calls_keep_their_scores(cuda, batch, tokens, heads, kept):
    """Without a workspace; those that have one and still keep them are pinned in tests/host/index_math_test.cpp."""
    assert bool(rules().keeps_scores(batch, tokens, heads)) == kept
    test_absorbed_backward_of_short_sequences(cuda, batch, tokens, heads)


@pytest.mark.parametrize("batch,tokens,heads", [(1, 1, 1), (3, 9, 2), (1, 513, 1), (2, 700, 3), (1, 1024, 2)])
def test_absorbed_backward_of_whole_key_blocks(cuda, batch, tokens, heads):
    """Calls whose query gradients have no room for partial results: without a workspace a workgroup walks all rows of its
    key block."""
    units = torch.cuda.get_device_properties(cuda).multi_processor_count
    assert not rules().keeps_scores(batch, tokens, heads) and rules().backward_ranges(batch, tokens, heads, units) == 0
    test_absorbed_backward_of_short_sequences(cuda, batch, tokens, heads)
