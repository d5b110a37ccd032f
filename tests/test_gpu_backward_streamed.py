"""GPU parity of the per-head backward on both sides of the size from which its gradient rows leave past the caches
(csrc/attn_bwd.hip, GRADIENT_STREAM_BYTES): dQ, dK and dV of 96 MiB together or a little less; and on both sides of the walks
(SHORT_WALK) from which dQ of 192 / 128 columns stays in them."""

import pytest
import torch

from dscuda_amd.harness import configs, ops
from oracle import attention_oracle as oracle
from parity import announce, assert_close_bf16

pytestmark = pytest.mark.gpu

LINE = 96 << 20


@pytest.mark.parametrize("seq,q_heads,kv_heads,dqk,dv,streamed", [
    (1535, 64, 64, 192, 128, False), (1537, 64, 64, 192, 128, True),   # last blocks of 127 keys and of one
    (2048, 64, 64, 128, 128, True), (1984, 64, 64, 128, 128, False),   # at the line itself
    (4096, 128, 16, 64, 64, False), (4928, 128, 16, 64, 64, True),
    (479, 20, 20, 192, 128, False), (480, 20, 20, 192, 128, False),
])
def test_gradients(cuda, seq, q_heads, kv_heads, dqk, dv, streamed):
    assert (2 * seq * (q_heads * dqk + kv_heads * (dqk + dv)) >= LINE) == streamed
    g = torch.Generator(device=cuda).manual_seed(seq)
    randn = lambda heads, dim: torch.randn(1, seq, heads, dim, device=cuda, generator=g).mul_(0.5).bfloat16()
    q, k, v, dout = randn(q_heads, dqk), randn(kv_heads, dqk), randn(kv_heads, dv), randn(q_heads, dv)
    scale = configs.c_float(dqk ** -0.5)
    announce("backward, streamed gradients", dict(T=seq, Hq=q_heads, Hkv=kv_heads, dqk=dqk, dv=dv))
    grads = tuple(torch.full_like(x, float("nan")) for x in (q, k, v))
    if dqk == dv:
        out, lse = ops.flash_forward(q, k, v, scale)
        workspace = ops.flash_backward_workspace(1, seq, q_heads, kv_heads, dqk)
        ops.flash_backward(dout, out, lse, q, k, v, scale, workspace, grads)
    else:
        out, lse = ops.mla_prefill_forward(q, k, v, scale)
        workspace = ops.mla_prefill_backward_workspace(1, seq, q_heads, dqk, dv)
        ops.mla_prefill_backward(dout, out, lse, q, k, v, scale, workspace, grads)
    torch.cuda.synchronize()
    assert all(torch.isfinite(x).all() for x in grads)
    sharing = q_heads // kv_heads
    pair = kv_heads - 1
    of_q = lambda x: x[:, :, pair * sharing:(pair + 1) * sharing].cpu()
    of_kv = lambda x: x[:, :, pair:pair + 1].cpu()
    expected = oracle.attention_backward(of_q(dout), of_q(out), lse[:, pair * sharing:(pair + 1) * sharing].cpu(), of_q(q), of_kv(k),
                                         of_kv(v), scale)
    for name, actual, reference in zip(("dQ", "dK", "dV"), (of_q(grads[0]), of_kv(grads[1]), of_kv(grads[2])), expected):
        assert_close_bf16(name, actual, reference)
