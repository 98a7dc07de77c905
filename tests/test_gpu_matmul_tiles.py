"""The tile GEMM kernels at the shapes where they can go wrong: one row or column past a tile,
a k-tile remainder of one chunk or one element, K shorter than the split over wave groups,
single rows and columns, views with their own strides, and C at odd element offsets.  Every
kernel of every input type runs (asserted from the dispatched kernel names).  fp32
accumulators of fp16 / bf16 / fp32 inputs are held to the bound of any summation order,
K * 2^-23 * (|A| @ |B|) (a product of two 16-bit values is exact in fp32; fp32 inputs round
each product too), plus the output's one rounding; int8 is exact."""
import pytest
import torch

from pyasc_amd import kernels

pytestmark = pytest.mark.gpu

ROUND = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
# one shape per kernel (its dispatch) and edge; N, K whole chunks
ALIGNED = [(1, 64, 64), (33, 40, 8), (31, 520, 1032), (17, 8200, 136), (65, 2056, 264), (100, 4096, 4096),
           (129, 1032, 40), (255, 2048, 200), (257, 4104, 520), (513, 4104, 1032), (333, 11008, 264),
           (1999, 4096, 72), (150, 4096, 4096), (1025, 2056, 136), (3001, 3008, 200), (2049, 4104, 4104)]
# nothing aligned
ODD = [(1, 1, 1), (3, 5, 7), (33, 31, 33), (64, 65, 1001), (127, 129, 63), (200, 301, 35), (200, 1001, 35), (257, 1001, 65),
       (1001, 2003, 131), (3001, 2999, 97), (260, 261, 401)]
SEEN = set()


def _check(c, a, b, bias, act, alpha):
    # fp64 on the GPU: the exact product of the rounded inputs to ~2^-53
    ad, bd = a.double(), b.double()
    exact = ad @ bd
    bound = (a.shape[1] + 2) * 2.0 ** -23 * (ad.abs() @ bd.abs())
    if bias is not None:
        exact += bias.double()
        bound += 2.0 ** -23 * exact.abs()
    if act == "relu":
        exact = exact.clamp(min=0)
    elif act == "leaky":
        exact = torch.where(exact >= 0, exact, exact * alpha)
    bound = bound + ROUND[c.dtype] * (exact.abs() + bound) + 1e-7
    over = (c.double() - exact).abs() > bound
    assert not over.any(), f"{int(over.sum())} of {over.numel()} elements off, first {over.nonzero()[0].tolist()}"


@pytest.mark.parametrize("shape", ALIGNED + ODD, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
def test_tiles_against_fp64(device, dtype, shape):
    M, N, K = shape
    g = torch.Generator(device=device).manual_seed(M * 7 + N * 3 + K)
    a = torch.randn((M, K), generator=g, device=device).to(dtype)
    b = torch.randn((K, N), generator=g, device=device).to(dtype)
    i = (ALIGNED + ODD).index(shape)
    out = [dtype, torch.float32, torch.bfloat16, torch.float16][i % 4]
    act = ["none", "relu", "leaky"][i % 3]
    bias = torch.randn(N, generator=g, device=device) if i % 2 else None
    c = torch.full((M, N), 7.0, dtype=out, device=device)
    kw = dict(relu=act == "relu", bias=bias, leaky_alpha=0.25 if act == "leaky" else None)
    SEEN.add(kernels.matmul_dispatch(a, b, c, **kw).kernel.decode())
    kernels.matmul(a, b, c, **kw)
    torch.cuda.synchronize()
    _check(c, a, b, bias, act, 0.25)


@pytest.mark.parametrize("shape", [(100, 264, 136), (300, 520, 72), (65, 130, 33)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_views_keep_their_surroundings(device, dtype, shape):
    # operands and C inside larger tensors, the values around them NaN: none may reach C, and
    # nothing around C may change; C starts at an odd element
    M, N, K = shape
    g = torch.Generator(device=device).manual_seed(1)
    big_a = torch.full((M + 2, K + 24), float("nan"), dtype=dtype, device=device)
    big_b = torch.full((K + 2, N + 40), float("nan"), dtype=dtype, device=device)
    a, b = big_a[1:M + 1, 8:8 + K], big_b[1:K + 1, 16:16 + N]
    a.copy_(torch.randn((M, K), generator=g, device=device))
    b.copy_(torch.randn((K, N), generator=g, device=device))
    big_c = torch.full((M + 2, N + 9), 5.0, dtype=torch.float32, device=device)
    c = big_c[1:M + 1, 3:3 + N]
    kernels.matmul(a, b, c)
    torch.cuda.synchronize()
    _check(c, a, b, None, "none", 0.0)
    around = big_c.clone()
    around[1:M + 1, 3:3 + N] = 5.0
    assert (around == 5.0).all()


def test_nan_and_inf_stay_in_their_rows_and_columns(device):
    # a k-tile remainder must not multiply values of the next row, and infinities pass through
    a = torch.randn((70, 72), device=device).to(torch.bfloat16)
    b = torch.randn((72, 136), device=device).to(torch.bfloat16)
    a[5, 3], a[9, 71] = float("inf"), float("nan")
    c = torch.empty((70, 136), device=device)
    kernels.matmul(a, b, c, relu=False)
    torch.cuda.synchronize()
    bad = ~torch.isfinite(c).all(dim=1)
    assert bad.nonzero().flatten().tolist() == [5, 9] and torch.isnan(c[9]).all()
    assert torch.equal(torch.isinf(c[5]), b[3] != 0)


I8 = [(1, 64, 64), (33, 48, 16), (31, 528, 1040), (16, 11008, 144), (129, 2064, 272), (257, 4112, 528), (333, 11008, 272),
      (600, 4096, 144), (1999, 4096, 80), (3000, 11008, 80), (150, 4096, 4096), (1, 1, 1), (5, 3, 7), (65, 33, 1001),
      (127, 257, 129), (257, 1001, 129), (347, 10080, 329), (1001, 3001, 67), (3001, 4999, 35), (2049, 4112, 4112)]


@pytest.mark.parametrize("shape", I8, ids=lambda s: "x".join(map(str, s)))
def test_int8_tiles_are_exact(device, shape):
    M, N, K = shape
    g = torch.Generator(device=device).manual_seed(M + N + K)
    a, b = (torch.randint(-128, 128, s, generator=g, device=device, dtype=torch.int8) for s in ((M, K), (K, N)))
    scale = torch.rand(N, generator=g, device=device) * 1e-3 + 1e-4
    acc = torch.full((M, N), 7, dtype=torch.int32, device=device)
    deq = torch.full((M, N), 7.0, dtype=torch.float16, device=device)
    SEEN.add(kernels.matmul_i8_dispatch(a, b, acc).kernel.decode())
    kernels.matmul_i8(a, b, acc)
    kernels.matmul_i8(a, b, deq, scale=scale, trunc19=M % 2 == 1)
    torch.cuda.synchronize()
    exact = (a.double() @ b.double())  # integers below 2^53
    assert torch.equal(acc.double(), exact)
    s = (scale.view(torch.int32) & -8192).view(torch.float32) if M % 2 == 1 else scale
    assert torch.equal(deq, (exact.float() * s).half())


def test_every_tile_kernel_ran(device):
    from pyasc_amd.launchers import MATMUL_CO_FUNCTIONS, MATMUL_I8_CO_FUNCTIONS
    assert {n for n in MATMUL_CO_FUNCTIONS + MATMUL_I8_CO_FUNCTIONS if "_tile_" in n} <= SEEN


@pytest.mark.parametrize("shape", [(1, 64, 4), (8, 1024, 512), (16, 16, 16), (64, 64, 64), (100, 100, 128), (256, 256, 64),
                                   (512, 512, 16), (260, 261, 57), (300, 257, 256), (9, 11007, 101)],
                         ids=lambda s: "x".join(map(str, s)))
def test_short_f32_products_take_blocks(device, shape):
    # 16x16 blocks where a tile's start takes longer than the product
    M, N, K = shape
    g = torch.Generator(device=device).manual_seed(M + N + K)
    a = torch.randn((M, K), generator=g, device=device)
    b = torch.randn((K, N), generator=g, device=device)
    bias = torch.randn(N, generator=g, device=device)
    c = torch.full((M, N), 7.0, device=device)
    kw = dict(bias=bias, leaky_alpha=0.25)
    assert kernels.matmul_dispatch(a, b, c, **kw).kernel.decode() == "asc2_mm_f32_mfma_f32"
    kernels.matmul(a, b, c, **kw)
    torch.cuda.synchronize()
    _check(c, a, b, bias, "leaky", 0.25)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("M,N", [(1000, 256), (300, 64), (513, 200), (1, 256)])
def test_product_in_place_of_a(device, dtype, M, N):
    # up to 256 columns: a workgroup of the 256x256 tiles' kernels reads whole rows before it writes them
    g = torch.Generator(device=device).manual_seed(M + N)
    a = torch.randn((M, N), generator=g, device=device).to(dtype)
    b = (torch.randn((N, N), generator=g, device=device) / N ** 0.5).to(dtype)
    x = a.clone()
    assert "_tile_" not in kernels.matmul_dispatch(x, b, x).kernel.decode()
    kernels.matmul(x, b, x)
    torch.cuda.synchronize()
    _check(x, a, b, None, "none", 0.0)
    # A and C side by side in one buffer share no memory
    buf = torch.full((M, 2 * N), 7.0, dtype=dtype, device=device)
    buf[:, :N] = a
    kernels.matmul(buf[:, :N], b, buf[:, N:])
    torch.cuda.synchronize()
    _check(buf[:, N:], a, b, None, "none", 0.0)
    assert torch.equal(buf[:, :N], a)
