"""Workspaces of launches on another stream than torch's current one, while the current stream
still has work queued on blocks that are already free again in its pool: the split reductions
and the chained matmul must neither disturb that work nor be disturbed by it."""
import ctypes

import pytest
import torch

from pyasc_amd import kernels

pytestmark = pytest.mark.gpu


def _busy_current_stream(device, sizes):
    """Queues, behind about 20 ms of other work, a fill and a copy of one block of each size
    (bytes), and frees the blocks: torch's pool of the current stream holds them at once."""
    torch.cuda._sleep(40_000_000)
    copies = []
    for n in sizes:
        block = torch.full((n,), 7, dtype=torch.uint8, device=device)
        copies.append(block.clone())
        del block
    return copies


@pytest.mark.parametrize("launch_on", ["side", "default"])
def test_reduction_beside_a_busy_stream(device, launch_on):
    x = torch.rand(16384, 100, device=device)
    want, out = torch.empty(100, device=device), torch.empty(100, device=device)
    kernels.reduce_f32(x, want, "sum", 0)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    stream, current = (side, torch.cuda.default_stream()) if launch_on == "side" else \
        (torch.cuda.default_stream(), side)
    with torch.cuda.stream(current):
        for _ in range(3):
            copies = _busy_current_stream(device, [12800, 65536, 4096])
            kernels.reduce_f32(x, out, "sum", 0, stream=stream)
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            assert all(bool((c == 7).all()) for c in copies)


def test_chained_matmul_beside_a_busy_stream(device):
    a = torch.randn(256, 128, device=device).to(torch.bfloat16)
    b = torch.randn(128, 128, device=device).to(torch.bfloat16)
    want, out = torch.empty(256, 128, device=device), torch.empty(256, 128, device=device)
    kernels.matmul_chained(a, b, want)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    for _ in range(3):
        copies = _busy_current_stream(device, [256 * 128 * 2, 65536])
        kernels.matmul_chained(a, b, out, stream=s)
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert all(bool((c == 7).all()) for c in copies)


def test_the_null_handle_is_the_default_stream(device):
    # an external stream of a null pointer would be one of torch's pool
    with torch.cuda.stream(torch.cuda.Stream()):
        w = kernels.workspace_on(0, 4096, torch.uint8, torch.device("cuda", torch.cuda.current_device()))
    x = torch.empty_like(w)  # the default stream's pool hands the freed block out again
    ptr = w.data_ptr()
    del w
    y = torch.empty(4096, dtype=torch.uint8, device=device)
    assert y.data_ptr() == ptr and x.data_ptr() != ptr


def _hip():
    """The HIP runtime that this process has loaded."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    hip.hipStreamBeginCapture.argtypes = [ctypes.c_void_p, ctypes.c_int]
    hip.hipStreamEndCapture.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)]
    hip.hipGraphInstantiate.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_void_p, ctypes.c_void_p,
                                        ctypes.c_void_p, ctypes.c_size_t]
    hip.hipGraphLaunch.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    hip.hipGraphExecDestroy.argtypes = hip.hipGraphDestroy.argtypes = [ctypes.c_void_p]
    return hip


@pytest.mark.parametrize("current", [True, False])
def test_reduction_in_a_graph_captured_without_torch(device, current):
    # the replays must not depend on memory that torch takes back when the call returns
    hip, relaxed = _hip(), 2
    x = torch.rand(16384, 100, device=device)
    out, want = torch.empty(100, device=device), torch.empty(100, device=device)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph, executable = ctypes.c_void_p(), ctypes.c_void_p()
    with torch.cuda.stream(s if current else torch.cuda.current_stream()):
        assert hip.hipStreamBeginCapture(s.cuda_stream, relaxed) == 0
        kernels.reduce_f32(x, out, "sum", 0, stream=None if current else s)
        assert hip.hipStreamEndCapture(s.cuda_stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(executable), graph, None, None, 0) == 0
    for _ in range(3):
        x.copy_(torch.rand(16384, 100, device=device))
        kernels.reduce_f32(x, want, "sum", 0)
        with torch.cuda.stream(s):  # whoever gets a workspace's memory next keeps it
            others = [torch.full((n,), 3.0, device=device) for n in (12800, 16384, 1000)]
        torch.cuda.synchronize()
        assert hip.hipGraphLaunch(executable, s.cuda_stream) == 0
        torch.cuda.synchronize()
        # sums of 16384 non-negative values in two orders
        assert ((out - want).abs() <= 2 * 16384 * 2.0 ** -24 * want).all()
        assert all(bool((o == 3.0).all()) for o in others)
        del others
    assert hip.hipGraphExecDestroy(executable) == 0 and hip.hipGraphDestroy(graph) == 0
