"""mla_absorb_query by quarters of the columns: chunks and token tiles cut at the edges, heads that no XCD order deals out,
strided and gapped results, and the last size before whole rows."""

import pytest
import torch

from dscuda_amd.harness import ops
from oracle import attention_oracle as oracle
from parity import announce, assert_close_bf16

pytestmark = pytest.mark.gpu


# more than 128 (token tiles x heads); one row in the last tile, one tile in the last chunk; 8 | heads and not
@pytest.mark.parametrize("tokens,heads", [(65, 128), (129, 65), (257, 40), (2049, 7), (5000, 2), (4225, 3), (9000, 1), (1000, 17)])
def test_absorb_query_by_quarters(cuda, tokens, heads):
    g = torch.Generator().manual_seed(61)
    weights = (torch.randn(heads, 256, 512, generator=g) * 0.06).bfloat16()
    query = (torch.randn(1, tokens, heads, 192, generator=g) * 0.5).bfloat16()
    announce("mla_absorb_query, quarters", dict(T=tokens, H=heads))
    packed = torch.full((1, tokens + 1, heads, 576), 7.0, device=cuda, dtype=torch.bfloat16)
    ops.mla_absorb_query(query.to(cuda)[..., :128], weights.to(cuda)[:, :128], out=packed[:, :tokens, :, :512])
    torch.cuda.synchronize()
    assert_close_bf16("q_latent", packed[:, :tokens, :, :512].cpu(), oracle.absorb_query(query[..., :128], weights[:, :128]))
    assert (packed[:, tokens:].float() == 7.0).all() and (packed[..., 512:].float() == 7.0).all()


# 144 MiB of results and more: one round of chunks of many heads, many chunks of few
@pytest.mark.parametrize("tokens,heads", [(1152, 128), (1153, 128), (18432, 8), (18433, 8), (147457, 1)])
def test_either_side_of_the_size_rule(cuda, tokens, heads):
    """A head's rows are the same bits whichever kernel forms them, in a buffer of rows with other columns behind them."""
    g = torch.Generator(device=cuda).manual_seed(67)
    weights = torch.randn(heads, 128, 512, device=cuda, generator=g).mul_(0.06).bfloat16()
    query = torch.randn(1, tokens, heads, 128, device=cuda, generator=g).mul_(0.5).bfloat16()
    announce("mla_absorb_query, size rule", dict(T=tokens, H=heads))
    packed = torch.full((1, tokens + 1, heads, 576), 7.0, device=cuda, dtype=torch.bfloat16)
    ops.mla_absorb_query(query, weights, out=packed[:, :tokens, :, :512])
    for first in range(0, tokens, (tokens + 3) // 4):   # a quarter of the tokens: the kernel by quarters of the columns
        part = ops.mla_absorb_query(query[:, first:first + (tokens + 3) // 4].contiguous(), weights)
        torch.cuda.synchronize()
        assert torch.equal(packed[:, first:min(first + (tokens + 3) // 4, tokens), :, :512], part)
    assert (packed[:, tokens:] == 7.0).all() and (packed[..., 512:] == 7.0).all()
