"""What the operators do with the workspaces their callers pass, on the host: the library is a stand-in that records its
calls, the operands are host tensors that say they are on a GPU."""

from types import SimpleNamespace

import pytest
import torch

from dscuda_amd.harness import ops


class OnGpu(torch.Tensor):
    is_cuda = property(lambda self: True)


def operand(*shape, dtype=torch.bfloat16):
    return torch.zeros(*shape, dtype=dtype).as_subclass(OnGpu)


@pytest.fixture
def calls(monkeypatch):
    """Names of the library functions that were called, in order."""
    names = []

    def function(name):
        def call(*arguments):
            names.append(name)
            return 0
        return call

    library = SimpleNamespace(lib=None, **{name: function(name) for name in (
        "backward", "backward_workspace", "backward_workspace_elements", "prefill_backward", "prefill_workspace", "decode",
        "decode_planned", "workspace")})
    monkeypatch.setattr(ops, "mla_library", lambda: library)
    monkeypatch.setattr(ops, "flash_library", lambda: library)
    monkeypatch.setattr(ops, "stream", lambda: 0)
    return names


def absorbed_backward(workspace):
    b, t, h = 1, 4, 2
    rows, lse = operand(b, t, h, 512), operand(b, h, t, dtype=torch.float32)
    return ops.mla_backward(rows, rows, lse, rows, operand(b, t, h, 64), operand(b, t, 512), operand(b, t, 64), 1.0,
                            workspace=workspace)


def prefill_backward(workspace):
    b, s, h = 1, 4, 2
    query, value = operand(b, s, h, 192), operand(b, s, h, 128)
    return ops.mla_prefill_backward(value, value, operand(b, h, s, dtype=torch.float32), query, query, value, 1.0, workspace)


def flash_backward(workspace):
    rows = operand(1, 64, 2, 64)
    return ops.flash_backward(rows, rows, operand(1, 2, 64, dtype=torch.float32), rows, rows, rows, 1.0, workspace)


def decode_operands():
    return operand(2, 1, 4, 576), operand(3, 64, 1, 576), operand(2, 2, dtype=torch.int32), operand(2, dtype=torch.int32)


def decode(workspace):
    return ops.mla_decode(*decode_operands(), 1.0, workspace=workspace)


def decode_planned(workspace):
    return ops.mla_decode_planned(*decode_operands(), operand(8, dtype=torch.int32), 1.0, workspace=workspace)


@pytest.mark.parametrize("call", [absorbed_backward, prefill_backward, flash_backward, decode, decode_planned])
def test_a_workspace_is_contiguous_gpu_memory(calls, call):
    """The kernels write through its pointer: memory of the host, or a view whose elements lie apart, is refused."""
    for workspace in (torch.zeros(64), operand(64, dtype=torch.float32)[::2]):
        with pytest.raises(RuntimeError, match="need"):
            call(workspace)
    assert calls == []
    call(operand(64, dtype=torch.float32))
    call(operand(0, dtype=torch.float32))
    assert len(calls) == 2


def test_an_empty_workspace_stands_for_none(calls):
    """The library's own backward without a workspace, and no question about the size of one."""
    absorbed_backward(operand(0, dtype=torch.float32))
    assert calls == ["backward"]
    absorbed_backward(operand(64, dtype=torch.float32))
    assert calls == ["backward", "backward_workspace"]


def test_a_large_workspace_is_not_asked_for_where_the_memory_is_short(calls, monkeypatch):
    """An allocation that fails gives all of torch's cached blocks back first: the call runs without, and nothing is tried."""
    ops.mla_library().backward_workspace_elements = lambda *shape: 1 << 28   # 1 GiB
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (100 << 20, 288 << 30))
    cached = [800 << 20]
    monkeypatch.setattr(torch.cuda, "memory_stats", lambda device: {
        "reserved_bytes.all.current": 10 << 30, "allocated_bytes.all.current": (10 << 30) - cached[0]})
    tried = []
    allocate = torch.empty

    def empty(*shape, **options):
        if shape == (1 << 28,):
            tried.append(shape)
            return operand(64, dtype=torch.float32)
        return allocate(*shape, **options)

    monkeypatch.setattr(torch, "empty", empty)
    absorbed_backward(None)
    assert calls == ["backward"] and not tried
    cached[0] = 950 << 20   # the cache holds what is missing
    absorbed_backward(None)
    assert calls == ["backward", "backward_workspace"] and len(tried) == 1
