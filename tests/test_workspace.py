"""The per-device attention workspace: what is allocated, kept and given up,
with the allocator stubbed (no GPU)."""
import weakref

import pytest
import torch

from nanovllm_self_amd.layers import attention as LA

CPU = torch.device("cpu")


class _Memory:
    """torch.empty with at most `room` bytes a tensor; keeps the sizes asked for."""

    def __init__(self, room):
        self.room, self.asked, self.empty = room, [], torch.empty

    def __call__(self, n, dtype, device):
        self.asked.append(n)
        if n > self.room:
            raise torch.cuda.OutOfMemoryError("stub")
        return self.empty(n, dtype=dtype, device=device)


@pytest.fixture
def memory(monkeypatch):
    for name in ("_workspaces", "_no_room", "_captured_workspaces"):
        monkeypatch.setattr(LA, name, {}, raising=False)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    mem = _Memory(1 << 20)
    monkeypatch.setattr(torch, "empty", mem)
    return mem


def test_no_memory_for_the_optional_bytes(memory):
    """The call is served without them, by the buffer that is there or by one
    of the bytes it cannot do without; as many are not asked for again."""
    assert LA.attention_workspace(CPU, 1000, 1 << 20).numel() == 1000
    assert memory.asked == [1000 + (1 << 20), 1000]
    there = LA.attention_workspace(CPU, 1000)
    assert LA.attention_workspace(CPU, 900, 2 << 20) is there
    assert LA.attention_workspace(CPU, 1000, 1 << 20) is there
    assert len(memory.asked) == 2
    assert LA.attention_workspace(CPU, 1000, 500).numel() == 1500  # fewer: asked for, and there
    assert LA.attention_workspace(CPU, 3000, 1 << 20).numel() == 3000
    with pytest.raises(torch.cuda.OutOfMemoryError):
        LA.attention_workspace(CPU, 2 << 20)
    assert LA.attention_workspace(CPU, 3000).numel() == 3000


def test_reserve_asks_for_the_optional_bytes_again(memory):
    memory.room = 16 << 20
    args = (6, 300, 16384, 32, CPU, 8)
    LA.reserve_attention_workspace(*args)
    without = LA._workspaces[CPU].numel()
    assert memory.asked[0] > memory.room and memory.asked[1:] == [without]
    memory.room = 1 << 30
    LA.reserve_attention_workspace(*args)
    assert LA._workspaces[CPU].numel() == memory.asked[0]


def test_captured_buffers_stay_and_eager_calls_grow(memory, monkeypatch):
    """A buffer that a captured call used outlives its replacement; calls
    outside a capture get the optional bytes whatever was captured before."""
    LA.attention_workspace(CPU, 1000)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    first = LA.attention_workspace(CPU, 800, 500)  # as it is, without the optional bytes
    assert first.numel() == 1000
    with pytest.raises(RuntimeError, match="too small inside graph capture"):
        LA.attention_workspace(CPU, 1001)
    assert LA.attention_workspace(CPU, 900) is first
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    ref, address = weakref.ref(first), first.data_ptr()
    del first
    grown = LA.attention_workspace(CPU, 800, 500)
    assert grown.numel() == 1300
    assert ref() is not None and ref().data_ptr() == address
    last = LA.attention_workspace(CPU, 2000)  # the grown one, captured by nobody, is given up
    gone = weakref.ref(grown)
    del grown
    assert gone() is None and last.numel() == 2000


def test_reserved_buffer_grows_for_the_optional_bytes(memory):
    """A reservation for decode alone asks for no optional bytes; a prefill
    call after it gets them."""
    memory.room = 1 << 30
    LA.reserve_attention_workspace(64, 1, 8192, 32, CPU, 8)
    reserved = LA._workspaces[CPU].numel()
    assert LA.attention_workspace(CPU, reserved, 4096).numel() == reserved + 4096


def test_device_without_an_index_is_the_current_one(memory, monkeypatch):
    """reserve_attention_workspace(..., "cuda") reserves what calls on tensors
    of "cuda:1", the current device, look up."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    monkeypatch.setattr(torch, "empty", lambda n, dtype, device: torch.zeros(n, dtype=dtype))
    LA.reserve_attention_workspace(4, 1, 512, 16, "cuda", 8)
    assert list(LA._workspaces) == [torch.device("cuda:1")]
    assert LA.attention_workspace(torch.device("cuda:1"), 100) is LA._workspaces[torch.device("cuda:1")]
