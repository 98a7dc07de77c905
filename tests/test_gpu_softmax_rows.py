"""Softmax rows at the lengths where a body changes (16 lanes, a wave, a workgroup, registers
or two passes), with remainders of a vector, rows that start on any element, partial tiles
and fused blocks, and rows with infinities and NaN, against the fp64 softmax.  fp32: x - max is
rounded to fp32 (as the reference does), which alone moves exp by |x - max| * 2^-24 of its
value; exp, the sum, the reciprocal and the product add at most 8 ulp.  fp16: one ulp."""
import math

import pytest
import torch

from pyasc_amd import kernels

pytestmark = pytest.mark.gpu

F32 = [1, 3, 5, 255, 257, 511, 513, 1023, 1026, 2047, 4095, 4097, 8191, 8193, 12001, 16383, 16384, 16385, 16390, 24577,
       32768, 32769, 49152, 49153, 100003]
F16 = [1, 7, 8, 9, 16, 120, 121, 122, 128, 505, 506, 1000, 1017, 1018, 1024, 2047, 2049, 4095, 4097, 8191, 8195, 10007,
       16383, 16384, 16400, 24579, 32761, 32762, 65529, 65530, 100003]
MANY_F32 = [1, 5, 63, 64, 65, 129, 193, 257, 333, 385, 512, 513, 4099, 8191, 8193, 12001, 16383, 16384]
MANY_F16 = [3, 121, 122, 249, 250, 333, 377, 378, 505, 506, 1017, 1018, 1529, 1530, 2041, 2042, 3065, 3066, 4089, 4090,
            6137, 6138, 8185, 8186, 10007, 10234, 12281, 12282, 16377, 16378]


def _check(out, x, dtype):
    ref = torch.softmax(x.double(), dim=1)
    if dtype == torch.float32:
        depth = (x.double().amax(dim=1, keepdim=True) - x.double()).clamp(max=200.0)
        assert ((out.double() - ref).abs() <= ref * (depth + 16.0) * 2.0 ** -24 + 2.0 ** -148).all()
    else:  # one fp16 ulp: 2^-10 of the value, 2^-24 below the normal range
        assert ((out.double() - ref).abs() <= ref * 2.0 ** -10 + 2.0 ** -24).all()


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype,cols", [(torch.float32, c) for c in F32] + [(torch.float16, c) for c in F16])
def test_row_lengths(device, dtype, cols, offset):
    rows = 37 if cols < 5000 else 5
    _row_lengths(device, dtype, cols, offset, rows)


@pytest.mark.parametrize("dtype,cols", [(torch.float32, c) for c in MANY_F32] + [(torch.float16, c) for c in MANY_F16])
def test_many_rows(device, dtype, cols):
    # more rows than any of the rules on the number of rows asks for, not a multiple of a workgroup's
    _row_lengths(device, dtype, cols, 1, 2053)


def _row_lengths(device, dtype, cols, offset, rows):
    g = torch.Generator(device=device).manual_seed(cols)
    x = torch.empty(rows * cols + offset, dtype=dtype, device=device)[offset:].view(rows, cols)
    x.copy_(torch.randn((rows, cols), generator=g, device=device) * 4)
    buf = torch.full((rows * cols + offset + 8,), 7.0, dtype=dtype, device=device)
    out = buf[offset:offset + rows * cols].view(rows, cols)
    kernels.softmax_rows(x, out, rows, cols, cols, 16)
    torch.cuda.synchronize()
    _check(out, x, dtype)
    assert (buf[:offset] == 7.0).all() and (buf[offset + rows * cols:] == 7.0).all()


@pytest.mark.parametrize("rows", [1, 3, 1024, 1025])
@pytest.mark.parametrize("cols", [1, 63, 64, 65, 127, 128, 129, 255, 257, 511, 512, 513, 767, 769, 1016, 1017, 1018])
def test_few_half_rows(device, cols, rows):
    # rows taken by elements or by vectors, by their number, length and alignment
    for offset in (0, 1, 4):
        _row_lengths(device, torch.float16, cols, offset, rows)


@pytest.mark.parametrize("cols", [64, 100, 192, 200, 256, 384, 400, 512])
def test_short_rows_round_their_sum_once(device, cols):
    # Rows of nearly equal values: what a row's results have in common is the rounding of the sum
    # and of its reciprocal.  One rounding each has variances 1 / m^2 + m^2 / 4 <= 1.25 for a sum of
    # mantissa m, in units of (2^-24)^2 / 3; chains of up to 8 additions in 16 lanes add at most
    # 16 * (1 + 4 + ... + 64) / 64 / 256.  A tree that rounds at every level has 1/2 + 1/4 + 1/8 more.
    x = torch.randn((8192, cols), generator=torch.Generator(device=device).manual_seed(cols), device=device) * 0.1
    out = torch.empty_like(x)
    kernels.softmax_rows(x, out, 8192, cols, cols, 16)
    ref = torch.softmax(x.double(), dim=1)
    scale = (out.double() / ref).mean(dim=1) - 1  # what a row's results have in common
    assert scale.square().mean().sqrt().item() <= 2.0 ** -24 * ((1.25 + 16 * 204 / 64 / 256) / 3) ** 0.5


@pytest.mark.parametrize("dtype,cols,tile", [(torch.float32, 20000, 17001), (torch.float16, 20000, 17001),
                                             (torch.float16, 300, 77), (torch.float32, 300, 77)])
def test_partial_tiles_and_fused_blocks(device, dtype, cols, tile):
    x = (torch.randn((90, cols), device=device) * 3).to(dtype)
    out = torch.full((90, cols), 7.0, dtype=dtype, device=device)
    kernels.softmax_rows(x, out, 90, cols, tile, 16)
    torch.cuda.synchronize()
    _check(out[:, :tile], x[:, :tile], dtype)
    assert (out[:, tile:] == 7.0).all()
    out.fill_(7.0)
    kernels.softmax_blocks(x, out, 90, cols, 5, 16)  # rows [0, 80)
    torch.cuda.synchronize()
    _check(out[:80], x[:80], dtype)
    assert (out[80:] == 7.0).all()


def test_more_rows_than_workgroups(device):
    # the fp16 launch stops at 65536 workgroups; rows beyond are strided over
    for cols, rows in ((16, 1100003), (506, 262201), (4100, 65601)):
        x = torch.randn((rows, cols), device=device).half()
        out = torch.empty_like(x)
        kernels.softmax_rows(x, out, rows, cols, cols, 16)
        torch.cuda.synchronize()
        _check(out, x, torch.float16)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("cols", [100, 700, 5000, 12001, 40003])
def test_infinities_and_nan(device, dtype, cols):
    x = torch.randn((7, cols), device=device).to(dtype)
    x[0, 5] = float("-inf")           # ignored
    x[1] = float("-inf")              # all -inf: NaN
    x[2, cols // 2] = float("nan")    # NaN everywhere
    x[3, cols - 1] = float("inf")     # NaN everywhere
    x[4, 1:] = float("-inf")          # one finite element takes everything
    x[5] = 3.0
    x[6, ::2] = -60000.0 if dtype == torch.float16 else -1e30
    out = torch.empty_like(x)
    kernels.softmax_rows(x, out, 7, cols, cols, 16)
    torch.cuda.synchronize()
    ref = torch.softmax(x.double(), dim=1)
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    for r in (0, 4, 5, 6):
        _check(out[r:r + 1], x[r:r + 1], dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("short", [0, 3, 9, 20000])
def test_longest_rows(device, dtype, short):
    # rows whose vectors and chunks end at or past 2^31 elements, starting on an odd element: all of
    # the sum comes from the two ends, the rest is 0, and nothing around the row changes
    cols = 2 ** 31 - 1 - short
    x = torch.full((cols + 1,), -200.0, dtype=dtype, device=device)[1:]
    x[0], x[-1] = 11.0, 10.0
    buf = torch.full((cols + 2,), 7.0, dtype=dtype, device=device)
    out = buf[1:-1]
    kernels.softmax_rows(x, out, 1, cols, cols, 16)
    torch.cuda.synchronize()
    for at, want in ((0, 1 / (1 + math.exp(-1.0))), (-1, 1 / (1 + math.exp(1.0)))):
        assert abs(out[at].item() - want) <= want * (2.0 ** -10 if dtype == torch.float16 else 17 * 2.0 ** -24), at
    assert (out[1:-1] == 0).all() and buf[0] == 7.0 and buf[-1] == 7.0
