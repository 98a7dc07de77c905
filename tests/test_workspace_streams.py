"""Workspaces belong to the launch stream, checked without a GPU: torch's allocator serves a
block from the pool of the stream that is current when it is asked, and orders the block's
reuse on that stream only.  So whatever stream a call launches on has to be torch's current one
while its workspace is allocated, and torch's current stream is the caller's again afterwards."""
import contextlib
from types import SimpleNamespace

import pytest
import torch

from pyasc_amd import _native, kernels, launchers

CURRENT, OTHER = 0x1000, 0x2000
DEVICE = torch.device("cpu")


@pytest.fixture
def streams(monkeypatch):
    """torch's stream state as a list of handles (the last is current), the stream that each
    workspace was allocated under, and the handle that each native call was launched on."""
    state = SimpleNamespace(current=[CURRENT], allocated=[], launched=[])

    @contextlib.contextmanager
    def use(stream):
        state.current.append(stream.cuda_stream)
        yield
        state.current.pop()

    monkeypatch.setattr(torch.cuda, "default_stream", lambda device=None: SimpleNamespace(cuda_stream=0))
    # as torch's: a null pointer is no external stream but asks for one of the pool's
    monkeypatch.setattr(torch.cuda, "ExternalStream", lambda ptr, device=None: SimpleNamespace(
        cuda_stream=ptr or 0xBAD))
    monkeypatch.setattr(torch.cuda, "stream", use)
    state.capturing = set()
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state.current[-1] in state.capturing)
    monkeypatch.setattr(_native, "current_stream_handle", lambda device=None: state.current[-1])
    real_empty = torch.empty

    def empty(*args, **kwargs):
        state.allocated.append(state.current[-1])
        return real_empty(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", empty)
    monkeypatch.setattr(_native, "call", lambda name, *args: state.launched.append((name, args[-1])))
    monkeypatch.setattr(kernels, "_device_tensor", lambda t, name: t)
    return state


@pytest.mark.parametrize("stream,handle", [(None, CURRENT), (CURRENT, CURRENT), (OTHER, OTHER), (0, 0)])
@pytest.mark.parametrize("dim", [0, None])
def test_reduction_workspace(streams, stream, handle, dim):
    x, out = torch.zeros(8192, 64), torch.zeros(64 if dim == 0 else 1)
    streams.allocated.clear()
    kernels.reduce_f32(x, out, "sum", dim, stream=stream)
    assert streams.launched == [("asc_reduce_f32_ws", handle)]
    assert streams.allocated == [handle] and streams.current == [CURRENT]


@pytest.mark.parametrize("stream,handle", [(None, CURRENT), (OTHER, OTHER), (0, 0)])
def test_chained_matmul_workspace(streams, stream, handle):
    a, b, c = torch.zeros(8, 16, dtype=torch.float16), torch.zeros(16, 16, dtype=torch.float16), torch.zeros(8, 16)
    streams.allocated.clear()
    kernels.matmul_chained(a, b, c, stream=stream)
    assert streams.launched == [("asc_matmul_chained", handle)]
    assert streams.allocated == [handle] and streams.current == [CURRENT]


@pytest.mark.parametrize("handle", [CURRENT, OTHER, 0])
def test_chained_launch_intermediate(streams, handle):
    call = SimpleNamespace(stream=handle, consts={"dtype": torch.float32, "a_shape": (8, 16), "b_shape": (16, 16),
                                                  "c_shape": (8, 16)},
                           args={"a_ptr": torch.zeros(8, 16), "b_ptr": torch.zeros(16, 16),
                                 "c_ptr": torch.zeros(8, 16)})
    seen = []
    streams.allocated.clear()
    launchers._chained_body(call, lambda a, b, c, stream: seen.append((tuple(c.shape), stream)))
    assert seen == [((8, 16), handle)] * 2
    assert streams.allocated == [handle] and streams.current == [CURRENT]


@pytest.mark.parametrize("stream,handle", [(None, CURRENT), (OTHER, OTHER)])
@pytest.mark.parametrize("pool,entry", [((0, 0), "asc_reduce_f32"), ((1, 0), "asc_reduce_f32_ws"),
                                        (None, "asc_reduce_f32")])
def test_reduction_under_capture(streams, monkeypatch, stream, handle, pool, entry):
    # a graph's replays outlive the call: only a workspace in the graph's own pool may be recorded
    segment = {"address": 0, "total_size": 1 << 62}
    monkeypatch.setattr(torch.cuda, "memory_snapshot", lambda: [
        segment if pool is None else {**segment, "segment_pool_id": pool}])
    monkeypatch.setattr(torch.cuda, "get_allocator_backend", lambda: "native")
    x, out = torch.zeros(8192, 64), torch.zeros(64)
    streams.capturing = {handle}
    kernels.reduce_f32(x, out, "sum", 0, stream=stream)
    streams.capturing = {CURRENT, OTHER} - {handle}  # another stream's capture is no concern
    kernels.reduce_f32(x, out, "sum", 0, stream=stream)
    assert streams.launched == [(entry, handle), ("asc_reduce_f32_ws", handle)]
    assert streams.current == [CURRENT]
