"""The un-absorb as a stream of token tiles (csrc/mla_projection.hip): heads whose tokens end inside a tile, one, two, three and
many tiles a workgroup, chunks of a head of unequal length, more heads than compute units, rows apart in wider tensors."""

import pytest
import torch

from dscuda_amd.harness import ops
from oracle import attention_oracle as oracle
from parity import announce, assert_close_bf16


# most a workgroup has: one tile; two, the last of one token; three; 33 tiles; chunks of two tiles and a last one of one;
# two rounds of heads
@pytest.mark.gpu
@pytest.mark.parametrize("tokens,heads", [(32, 129), (33, 150), (96, 200), (65, 256), (1037, 200), (1000, 16), (1025, 33), (2049, 5), (70, 300), (129, 1),
                                          (4001, 4), (3000, 3), (2200, 16), (2200, 17)])   # runs of an XCD, of unequal length; none
def test_unabsorb_output(cuda, tokens, heads):
    g = torch.Generator().manual_seed(tokens + heads)
    wkv_b = (torch.randn(heads, 256, 512, generator=g) * 0.06).bfloat16()
    wide = (torch.randn(1, tokens, heads, 576, generator=g) * 0.5).bfloat16()
    announce("mla_unabsorb_output, stream", dict(T=tokens, H=heads))
    out = torch.full((1, tokens + 1, heads, 136), 7.0, device=cuda, dtype=torch.bfloat16)
    on_gpu = wide.to(cuda)
    ops.mla_unabsorb_output(on_gpu[..., :512], wkv_b.to(cuda)[:, 128:], out=out[:, :tokens, :, :128])
    dense = ops.mla_unabsorb_output(on_gpu[..., :512].contiguous(), wkv_b.to(cuda)[:, 128:].contiguous())
    torch.cuda.synchronize()
    assert (out[:, tokens:].float() == 7.0).all() and (out[..., 128:].float() == 7.0).all()
    assert torch.equal(out[:, :tokens, :, :128], dense)
    assert_close_bf16("output", dense.cpu(), oracle.unabsorb_output(wide[..., :512], wkv_b[:, 128:]))
