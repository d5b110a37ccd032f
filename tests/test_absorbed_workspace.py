"""The absorbed backward with a workspace (dS kept for the query gradients, slots for partial key gradients): its size
on the host, and on the GPU the gradients with and without one at the edges of tiles, blocks and items."""

import ctypes
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from dscuda_amd.harness import configs
from dscuda_amd.harness.common import I, bind, library
from dispatch_rules import rules
from oracle import attention_oracle as oracle
from parity import announce, assert_close_bf16


def elements(batch, tokens, heads, rank=512):
    return bind(library("mla"), "dscuda_mla_backward_workspace_elements", [I] * 5, ctypes.c_size_t)(
        batch, tokens, heads, rank, 64)


def kept_bytes(tokens, heads):
    """dS of one batch element: 2 KB per 32 x 32 tile that a key block of 32 (or 64) keys visits."""
    row_tiles = -(-tokens * heads // 32)
    return max(sum(max(0, row_tiles - size * heads * block) for block in range(-(-tokens // (32 * size)))) * 2048 * size
               for size in (1, 2))


@pytest.mark.parametrize("batch,tokens,heads", [
    (1, 513, 8), (3, 700, 5), (1, 65, 128), (2, 4096, 16), (1, 512, 8), (1, 2048, 128), (1, 4096, 128), (240, 4096, 1),
    (60, 4096, 4), (4096, 33, 16), (512, 1, 1), (20, 4096, 1), (271, 352, 2)])
def test_size_holds_every_block_and_the_slots_that_are_used(batch, tokens, heads):
    """dS, and the slots that the call uses for partial key gradients, unless the latent query gradients hold any number."""
    slots = rules().workspace_slots(batch, tokens, heads)
    room = elements(batch, tokens, heads) * 4 - batch * kept_bytes(tokens, heads)
    most = 3 * 256 * 64 * 576 * 4
    assert room == (slots if batch * tokens * heads * 1024 < most else 0) and room <= most


def test_size_is_zero_or_bounded():
    assert elements(1, 0, 8) == 0 and elements(1, 64, 8, rank=256) == 0
    assert elements(1, 300, 4) == 0                       # P and dS are kept in the query gradients
    assert elements(1, 16384, 128) == 0                   # dS of one batch element beyond 4 GiB: formed twice instead
    for batch, tokens, heads in ((64, 4096, 32), (300, 4096, 1), (2000, 1500, 1), (64, 4096, 4), (100000, 33, 3)):
        assert 0 < elements(batch, tokens, heads) * 4 <= (4 << 30) + 114_000_000, (batch, tokens, heads)


@pytest.mark.parametrize("batch,tokens,heads,passes", [(64, 4096, 4, 2), (300, 4096, 1, 2), (2000, 1500, 1, 2), (65, 2048, 32, 3)])
def test_batch_elements_are_taken_in_equal_passes(batch, tokens, heads, passes):
    """dS beyond 4 GiB: no last pass of a few elements that leaves the chip idle (64 elements as 63 and one)."""
    each = kept_bytes(tokens, heads)
    assert -(-batch // ((4 << 30) // each)) == passes
    assert 0 <= elements(batch, tokens, heads) * 4 - -(-batch // passes) * each <= 114_000_000


@pytest.mark.parametrize("batch,tokens,heads", [
    (1, 1 << 30, 1 << 30), (1, 2**31 - 1, 2**31 - 1), (2**31 - 1, 2**31 - 1, 2**31 - 1), (1, 2**31 - 1, 31),
    (2**31 - 1, 1, 33), (1, 1, 2**31 - 1)])
def test_size_of_calls_beyond_any_memory(batch, tokens, heads):
    """Arithmetic that leaves 64 bits, or a grid that the call refuses: no size, and in a process of its own because a
    division by a size of zero ends it."""
    code = ("import ctypes\nfrom dscuda_amd.harness.common import I, bind, library\n"
            "query = bind(library('mla'), 'dscuda_mla_backward_workspace_elements', [I] * 5, ctypes.c_size_t)\n"
            f"print(query({batch}, {tokens}, {heads}, 512, 64))")
    result = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300,
                            cwd=Path(__file__).resolve().parents[1])
    assert (result.returncode, result.stdout.strip()) == (0, "0"), (result.returncode, result.stdout, result.stderr[-500:])


# rows that end inside a row tile, a 64- and a 128-row workgroup; key blocks of 64 cut at 1, 32, 33 keys; one head, and
# more heads than a workgroup has rows; ranges of 32-key blocks and items of 64-key blocks; several batch elements; key
# blocks walked whole, of one to twelve row tiles; the query product's rows of a workgroup and halves of its columns by the
# number of workgroups: 64 rows a batch element and one more, short walks and long ones
@pytest.mark.gpu
@pytest.mark.parametrize("batch,tokens,heads,interval_tiles", [
    (1, 17, 128, 0), (2, 33, 40, 0), (1, 513, 3, 0), (1, 545, 8, 0), (3, 600, 4, 0), (1, 200, 33, 0), (2, 320, 16, 0),
    (1, 1000, 1, 0), (1, 1025, 8, 0), (1, 130, 150, 0), (1, 1, 40, 0), (1, 187, 32, 0), (3, 9, 2, 0), (2, 700, 3, 0),
    (1, 1000, 33, 0), (40, 33, 5, 0), (3, 64, 1, 0), (34, 126, 3, 0), (2, 2, 17, 0), (1, 512, 8, 0), (2, 530, 16, 0), (1, 513, 3, 7), (2, 97, 40, 50), (1, 65, 128, 100),
    (300, 3, 7, 0), (165, 2, 17, 0), (57, 21, 11, 0), (3, 193, 15, 0), (300, 5, 13, 0)])
def test_gradients_with_and_without(cuda, batch, tokens, heads, interval_tiles):
    from dscuda_amd.harness import ops
    ql, qr, c, kr, scale = configs.mla_absorbed_inputs(batch, tokens, heads)
    g = torch.Generator().manual_seed(6)
    dout = (torch.randn(batch, tokens, heads, 512, generator=g) * (0.2 if heads < 16 else 0.05)).bfloat16()
    mask = oracle.causal_mask(tokens)
    out, lse = oracle.mla_forward(ql, qr, c, kr, scale, mask)
    operands = [x.to(cuda) for x in (dout, out, lse, ql, qr, c, kr)]
    announce("mla_backward, workspace", dict(B=batch, T=tokens, H=heads, tiles=interval_tiles))

    def gradients(workspace):
        grads = tuple(torch.full_like(x, float("nan")) for x in operands[3:])
        return ops.mla_backward(*operands, scale, grads, workspace)

    ops.mla_backward_set_key_interval_tiles(interval_tiles)
    try:
        runs = [gradients(torch.empty(0, device=cuda)), gradients(None)]
        # dS of one batch element alone (the others after it, slots in the query gradients), and a guard behind it
        one = kept_bytes(tokens, heads) // 4
        buffer = torch.full((one + 1024,), float("nan"), device=cuda)
        runs.append(gradients(buffer[:one]))
        torch.cuda.synchronize()
    finally:
        ops.mla_backward_set_key_interval_tiles(0)
    assert torch.isnan(buffer[one:]).all()
    expected = oracle.mla_backward_unrounded(dout, out, lse, ql, qr, c, kr, scale, mask)
    for run in runs:
        for name, actual, reference in zip(("dq_latent", "dq_rope", "dlatent", "dk_rope"), run, expected):
            assert_close_bf16(name, actual.cpu(), reference)


# 128 rows a workgroup (two row tiles a wave), 64 rows, 64 rows and half the columns; 64-key blocks by the library's own
# choice and forced
@pytest.mark.gpu
@pytest.mark.parametrize("batch,tokens,heads,interval_tiles", [
    (32, 1000, 1, 0), (16, 700, 3, 0), (20, 850, 1, 0), (2, 450, 3, 0), (32, 1000, 1, 9), (20, 850, 1, 9), (2, 450, 3, 9)])
def test_keys_that_are_not_finite_stay_with_the_rows_that_see_their_tile(cuda, batch, tokens, heads, interval_tiles):
    """A row that sees none of 32 keys gets the same query gradient whatever those keys hold."""
    from dscuda_amd.harness import ops
    g = torch.Generator(device=cuda).manual_seed(7)

    def randn(*shape, factor=0.25):
        return (torch.randn(shape, device=cuda, generator=g) * factor).bfloat16()

    ql, qr = randn(batch, tokens, heads, 512), randn(batch, tokens, heads, 64)
    latent, kr, dout = randn(batch, tokens, 512), randn(batch, tokens, 64), randn(batch, tokens, heads, 512, factor=0.1)
    scale = configs.c_float(576 ** -0.5)
    out, lse = ops.mla_forward(ql, qr, latent, kr, scale)
    announce("mla_backward, keys not finite", dict(B=batch, T=tokens, H=heads, tiles=interval_tiles))
    ops.mla_backward_set_key_interval_tiles(interval_tiles)
    try:
        assert ops.mla_backward_workspace(batch, tokens, heads, device=cuda) is not None
        expected = ops.mla_backward(dout, out, lse, ql, qr, latent, kr, scale)[:2]
        for key in (tokens // 64 * 32 + 9, tokens // 64 * 32 + 41):   # an even and an odd tile of keys
            latent_changed, kr_changed = latent.clone(), kr.clone()
            latent_changed[:, key], kr_changed[:, key] = float("inf"), float("nan")
            actual = ops.mla_backward(dout, out, lse, ql, qr, latent_changed, kr_changed, scale)[:2]
            for name, a, b in zip(("dq_latent", "dq_rope"), actual, expected):
                assert torch.equal(a[:, :key // 32 * 32], b[:, :key // 32 * 32]), (name, key)
                assert torch.isnan(a[:, key:].float()).all(), (name, key)
    finally:
        ops.mla_backward_set_key_interval_tiles(0)
