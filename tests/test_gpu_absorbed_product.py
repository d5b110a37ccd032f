"""The absorbed backward's query product with 128 rows and all columns a workgroup (csrc/mla_absorbed_product.hip): rows that
end inside a row tile, a wave's pair of them or a workgroup, workgroups whose row tiles see different numbers of key tiles."""

import pytest
import torch

from dscuda_amd.harness import configs, ops
from oracle import attention_oracle as oracle
from parity import announce, assert_close_bf16


# workgroups of 128 rows: 396 (every third of one row), 259, 344, 262, 262, 264, 1560 (dS of 0.65 GB)
@pytest.mark.gpu
@pytest.mark.parametrize("batch,tokens,heads", [(132, 257, 1), (1, 1001, 33), (43, 1000, 1), (1, 515, 65), (131, 85, 3), (4, 840, 10),
                                                 (60, 3300, 1)])
def test_query_gradients(cuda, batch, tokens, heads):
    ql, qr, c, kr, scale = configs.mla_absorbed_inputs(batch, tokens, heads)
    g = torch.Generator().manual_seed(6)
    dout = (torch.randn(batch, tokens, heads, 512, generator=g) * (0.2 if heads < 16 else 0.05)).bfloat16()
    operands = [x.to(cuda) for x in (ql, qr, c, kr)]
    announce("mla_backward, query product", dict(B=batch, T=tokens, H=heads))
    out, lse = ops.mla_forward(*operands, scale)
    grads = tuple(torch.full_like(x, float("nan")) for x in operands)
    ops.mla_backward(dout.to(cuda), out, lse, *operands, scale, grads)
    torch.cuda.synchronize()
    some = sorted({0, batch // 2, batch - 1})
    expected = oracle.mla_backward_unrounded(dout[some], out.cpu()[some], lse.cpu()[some], ql[some], qr[some], c[some], kr[some],
                                             scale, oracle.causal_mask(tokens))
    for name, actual, reference in zip(("dq_latent", "dq_rope", "dlatent", "dk_rope"), grads, expected):
        assert_close_bf16(name, actual.cpu()[some], reference)
    assert all(torch.isfinite(x).all() for x in grads)
