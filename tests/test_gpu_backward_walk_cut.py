"""GPU parity of the backward where the walks of the key/value-gradient pass are cut into parts (choose_walk_cut): the
parts' fp32 sums are added in order and rounded once, so the tolerances are those of the uncut pass."""

import pytest
import torch

from dscuda_amd.harness import configs, ops
from oracle import attention_oracle as oracle
from tests.dispatch_rules import rules
from tests.parity import announce, assert_close_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,seq,q_heads,kv_heads,dqk,dv", [
    (1, 769, 16, 1, 64, 64),       # a last key block of one key; parts that begin and end inside a query head
    (3, 704, 6, 3, 64, 64),        # nine pairs: the plain workgroup order
    (1, 1000, 8, 8, 192, 128),     # one pair per XCD, the last tile ragged
    (2, 705, 3, 3, 192, 128),      # walks of 12 tiles, the shortest that are cut
    (1, 640, 8, 2, 128, 128),
    (1, 1024, 128, 32, 64, 64),    # more workgroups than run at once
])
def test_cut_walks(cuda, batch, seq, q_heads, kv_heads, dqk, dv):
    g = torch.Generator().manual_seed(71)
    randn = lambda heads, dim: (torch.randn(batch, seq, heads, dim, generator=g) * 0.5).bfloat16()
    q, k, v, dout = randn(q_heads, dqk), randn(kv_heads, dqk), randn(kv_heads, dv), randn(q_heads, dv)
    scale = configs.c_float(dqk ** -0.5)
    out_f, lse = oracle.causal_attention_forward(q, k, v, scale)
    out = out_f.bfloat16()
    announce("backward, cut walks", dict(B=batch, T=seq, Hq=q_heads, Hkv=kv_heads, dqk=dqk, dv=dv))
    operands = tuple(x.to(cuda) for x in (dout, out, lse, q, k, v))
    if dqk == dv:
        workspace = ops.flash_backward_workspace(batch, seq, q_heads, kv_heads, dqk)
    else:
        workspace = ops.mla_prefill_backward_workspace(batch, seq, q_heads, dqk, dv)
    assert rules().walks_are_cut(batch * kv_heads, seq, q_heads // kv_heads)
    key_blocks, tiles = (seq + 127) // 128, (seq + 63) // 64
    blocks = sum(tiles - 2 * kb for kb in range(key_blocks))
    assert workspace.numel() > batch * q_heads * (tiles * 128 + blocks * 4096)   # room for partial sums
    workspace.fill_(float("nan"))
    runs = []
    for _ in range(2):
        if dqk == dv:
            runs.append(ops.flash_backward(*operands, scale, workspace))
        else:
            runs.append(ops.mla_prefill_backward(*operands, scale, workspace))
    torch.cuda.synchronize()
    for name, first, second, expected in zip(("dQ", "dK", "dV"), *runs, oracle.attention_backward(dout, out, lse, q, k, v, scale)):
        assert torch.equal(first, second)
        assert_close_bf16(name, first.cpu(), expected)


def test_cut_walks_in_chunks_of_pairs(cuda):
    """T=8192 with 8 query heads per key/value head: the dS blocks of five pairs fill the budget, so the eight pairs run
    as five and three, every walk cut.  dQ equals that of one pair by itself; its dK and dV are the same sums in parts of
    other lengths, each rounded to bf16 once."""
    seq, sharing, kv_heads, dim = 8192, 8, 8, 64
    g = torch.Generator(device=cuda).manual_seed(72)
    randn = lambda heads: torch.randn(1, seq, heads, dim, device=cuda, generator=g).mul_(0.5).bfloat16()
    q, k, v, dout = randn(kv_heads * sharing), randn(kv_heads), randn(kv_heads), randn(kv_heads * sharing)
    scale = configs.c_float(dim ** -0.5)
    announce("backward, cut walks in chunks", dict(T=seq, Hq=kv_heads * sharing, Hkv=kv_heads, D=dim))
    out, lse = ops.flash_forward(q, k, v, scale)
    grads = ops.flash_backward(dout, out, lse, q, k, v, scale)
    for pair in (0, 4, 5, 7):
        heads, own = slice(sharing * pair, sharing * (pair + 1)), slice(pair, pair + 1)
        alone = ops.flash_backward(dout[:, :, heads].contiguous(), out[:, :, heads].contiguous(), lse[:, heads].contiguous(),
                                   q[:, :, heads].contiguous(), k[:, :, own].contiguous(), v[:, :, own].contiguous(), scale)
        torch.cuda.synchronize()
        assert torch.equal(grads[0][:, :, heads], alone[0])
        for whole, part in zip(grads[1:], alone[1:]):
            # one rounding apart at most (2**-8 of the value), and fp32 sums of 65536 terms
            torch.testing.assert_close(whole[:, :, own].float(), part.float(), rtol=2 ** -7, atol=1e-3)
