"""Reductions at the shapes where a kernel or its split changes: one column or row past a
workgroup's 64 columns, 64-row pass or unrolled step, rows that are not 16-byte aligned, few
long rows, few results over many elements (the split form and its second launch), and the
entry without a workspace.  max / min exact (torch), sums of non-negative values within the
bound of any order of fp32 additions, n * 2^-24 relative to the fp64 sum."""
import pytest
import torch

from pyasc_amd import _native, kernels

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (31, 33), (32, 31), (33, 32), (63, 5), (64, 64), (65, 65), (255, 130), (257, 127), (513, 100), (1023, 2049), (1024, 2048),
          (3, 100003), (16, 65536), (40, 70001), (5, 300001), (33, 262145), (65536, 16), (65537, 3), (16384, 4096),
          (9000, 31), (1, 262147), (4100, 1)]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_reduce_shapes(device, rows, cols, offset):
    g = torch.Generator(device=device).manual_seed(rows * 3 + cols)
    x = torch.rand(rows * cols + offset, generator=g, device=device)[offset:].view(rows, cols)
    x64 = x.double()
    for dim in (0, 1, None):
        shape = {0: cols, 1: rows, None: 3}[dim]
        terms = {0: rows, 1: cols, None: rows * cols}[dim]
        for op in ("sum", "max", "min"):
            out = torch.full((shape,), -7.0, device=device)
            kernels.reduce_f32(x, out, op, dim)
            if op == "sum":
                ref = (x64.sum() if dim is None else x64.sum(dim)).expand(shape)
                assert ((out.double() - ref).abs() <= terms * 2.0 ** -24 * ref).all(), (op, dim)
            else:
                f = torch.amax if op == "max" else torch.amin
                ref = (f(x) if dim is None else f(x, dim)).expand(shape)
                assert torch.equal(out, ref), (op, dim)


@pytest.mark.parametrize("dim", [0, -1])
def test_without_a_workspace_and_with_a_short_one(device, dim):
    rows, cols = 8192, 64
    x = torch.rand(rows, cols, device=device)
    n = cols if dim == 0 else 1
    need = _native.load_library().asc_reduce_f32_workspace(rows, cols, dim)
    assert 0 < need <= 65536
    plain, split = torch.empty(n, device=device), torch.empty(n, device=device)
    s = torch.cuda.current_stream().cuda_stream
    _native.call("asc_reduce_f32", 1, x.data_ptr(), plain.data_ptr(), rows, cols, dim, n, s)
    ws = torch.empty(need, dtype=torch.uint8, device=device)
    _native.call("asc_reduce_f32_ws", 1, x.data_ptr(), split.data_ptr(), rows, cols, dim, n, ws.data_ptr(), need, s)
    assert torch.equal(plain, split) and torch.equal(plain, x.amax(0) if dim == 0 else x.max().view(1))
    with pytest.raises(RuntimeError, match="the workspace holds"):
        _native.call("asc_reduce_f32_ws", 1, x.data_ptr(), split.data_ptr(), rows, cols, dim, n, ws.data_ptr(),
                     need - 4, s)


def test_special_values_and_product(device):
    x = torch.rand(5000, 70, device=device) + 0.5
    x[17, 3], x[4000, 3], x[300, 5], x[301, 6] = float("inf"), -float("inf"), float("nan"), -float("inf")
    out = torch.empty(70, device=device)
    kernels.reduce_f32(x, out, "max", 0)
    assert out[3] == float("inf") and torch.isfinite(out[5]) and torch.isfinite(out[6])  # maxNum skips NaN
    kernels.reduce_f32(x, out, "sum", 0)
    assert torch.isnan(out[3]) and torch.isnan(out[5]) and out[6] == -float("inf")
    y = 1.0 + 1e-4 * torch.randn(600, 1000, device=device)
    one = torch.empty(1, device=device)
    kernels.reduce_f32(y, one, "prod", None)
    ref = y.double().log().sum().exp()
    assert abs(one.item() / ref.item() - 1) < 600_000 * 2.0 ** -24


def test_split_reduction_on_a_side_stream_and_in_a_graph(device):
    x = torch.rand(16384, 100, device=device)
    want = torch.empty(100, device=device)
    kernels.reduce_f32(x, want, "sum", 0)
    out = torch.zeros(100, device=device)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    for _ in range(3):  # the workspace of one call may be reused by the next allocation
        kernels.reduce_f32(x, out, "sum", 0, stream=s)
        torch.rand(100000, device=device)
    s.synchronize()
    assert torch.equal(out, want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        kernels.reduce_f32(x, out, "sum", 0)
    for k in range(3):
        x.copy_(torch.rand(16384, 100, device=device))
        out.fill_(-1)
        g.replay()
        kernels.reduce_f32(x, want, "sum", 0)
        torch.cuda.synchronize()
        assert torch.equal(out, want), k


@pytest.mark.parametrize("rows,cols", [(512, 65536), (512, 3000), (300, 100003), (1024, 4096), (60000, 7),
                                       (60000, 17), (60000, 33), (60000, 64), (60000, 67)])
def test_row_sums_round_like_a_binary_tree(device, rows, cols):
    # the last additions of a sum carry its rounding error: in a binary tree their variances are
    # 1 + 1/2 + 1/4 + ... < 2 times that of one rounding, (2^-24)^2 / 3 relative at most.  A chain
    # over the parts of a row has 1 + (15/16)^2 + (14/16)^2 + ...
    x = torch.rand(rows, cols, generator=torch.Generator(device=device).manual_seed(cols), device=device)
    out = torch.empty(rows, device=device)
    kernels.reduce_f32(x, out, "sum", 1)
    ref = x.double().sum(1)
    rms = ((out.double() - ref) / ref).square().mean().sqrt().item()
    assert rms <= 2.0 ** -24 * (2 / 3) ** 0.5, rms


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("rows,cols", [(1, 262143), (2, 262144), (7, 65537), (8, 65536), (9, 262147), (15, 1001),
                                       (31, 270604), (16, 524292), (17, 524292), (33, 262145), (512, 4096), (512, 4095),
                                       (255, 2048), (257, 2048), (1023, 8184)])
def test_few_rows_and_row_lines(device, rows, cols, offset):
    # columns over one or four waves per workgroup, x above and below the size that is streamed,
    # 16-byte aligned or not, 1..7 rows behind a step of eight, and rows on both sides of the line
    # between a wave and a workgroup per row
    g = torch.Generator(device=device).manual_seed(rows + cols)
    x = torch.rand(rows * cols + offset, generator=g, device=device)[offset:].view(rows, cols)
    for dim, n in ((0, cols), (1, rows)):
        out = torch.full((n + 8,), -7.0, device=device)
        kernels.reduce_f32(x, out[4:n + 4], "sum", dim)
        ref = x.double().sum(dim)
        assert ((out[4:n + 4].double() - ref).abs() <= x.shape[dim] * 2.0 ** -24 * ref).all()
        kernels.reduce_f32(x, out[4:n + 4], "max", dim)
        assert torch.equal(out[4:n + 4], x.amax(dim))
        assert (out[:4] == -7.0).all() and (out[n + 4:] == -7.0).all()
