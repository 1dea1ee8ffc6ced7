"""Where a call under stream capture takes its workspace from.  Host logic, with torch's answers about the GPU replaced."""
import contextlib
import gc
import importlib
import weakref

import pytest
import torch

sub = importlib.import_module("amd-developer-challenge-2025_amd.submission")
CPU = torch.device("cpu")                       # its index, None, stands for the current device


@pytest.fixture
def capturing(monkeypatch):
    """A capture in progress; `pool` is the memory pool that allocations come from meanwhile ((0, 0): the ordinary one)."""
    state = {"pool": (0, 0), "on": True}
    monkeypatch.setattr(torch.cuda, "current_device", lambda: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["on"])
    monkeypatch.setattr(torch.cuda, "memory_snapshot", lambda *a: [{"segment_pool_id": state["pool"], "address": 0, "total_size": 1 << 62}])
    monkeypatch.setattr(sub, "_workspaces", {})
    monkeypatch.setattr(sub, "_held", {}, raising=False)
    return state


def test_a_capture_outside_a_torch_graph_keeps_the_buffers_it_saw(capturing):
    """The graph holds the address for as long as it lives: the buffer is never freed, not when a larger call outgrows it and
    not when the table drops its entry."""
    seen = []
    for nbytes in (1 << 20, 3 << 20, 64):
        ws = sub._workspace(CPU, nbytes, 7)
        assert ws.numel() >= nbytes
        seen.append(weakref.ref(ws.untyped_storage()))
        addr = ws.data_ptr()
        del ws
        assert sub._workspace(CPU, nbytes, 7).data_ptr() == addr
    capturing["on"] = False
    sub._workspace(CPU, 32 << 20, 7)
    for stream in range(100, 120):
        sub._workspace(CPU, 64, stream)
    gc.collect()
    assert all(s() is not None for s in seen)
    assert sum(t.numel() for t in sub._held[(None, 7)]) <= 2 * max(t.numel() for t in sub._held[(None, 7)])


def test_a_capture_outside_a_torch_graph_takes_the_buffer_an_eager_call_left(capturing):
    """No allocation of that size under such a capture: what the stream has is used, and kept from then on."""
    capturing["on"] = False
    addr = sub._workspace(CPU, 5 << 20, 3).data_ptr()
    capturing["on"] = True
    assert sub._workspace(CPU, 2 << 20, 3).data_ptr() == addr
    assert [t.data_ptr() for t in sub._held[(None, 3)]] == [addr]


def test_a_torch_graph_owns_its_buffers(capturing):
    capturing["pool"] = (4, 0)
    ref = weakref.ref(sub._workspace(CPU, 1 << 20, 7).untyped_storage())
    gc.collect()
    assert ref() is None and not sub._workspaces and not sub._held


def test_the_operands_device_is_asked(monkeypatch):
    """Capturing or not is a property of the stream the call goes to, which need not be the current device's."""
    now = [0]

    @contextlib.contextmanager
    def on(device):
        old, now[0] = now[0], device.index
        yield
        now[0] = old
    monkeypatch.setattr(torch.cuda, "current_device", lambda: now[0])
    monkeypatch.setattr(torch.cuda, "device", on)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: now[0] == 1)
    assert sub._capturing(torch.device("cuda", 1)) and not sub._capturing(torch.device("cuda", 0))
    now[0] = 1
    assert sub._capturing(torch.device("cuda", 1)) and not sub._capturing(torch.device("cuda", 0))
