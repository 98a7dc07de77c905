"""asc_matmul_dispatch and asc_matmul_i8_dispatch without a GPU: the launch the matmul entries
make.  Every dispatched launch covers C with whole tiles, fits one launch, carries the call's
arguments, uses the direct-to-LDS tiles only on operands made of 16-byte chunks, and fails
exactly where the plan of the 256x256-tile kernels fails.  Over many shapes the choice reaches
every tile kernel of the code objects."""
import ctypes
import random
import re
import struct

from hypothesis import given, settings, strategies as st

from pyasc_amd import _native
from pyasc_amd.launchers import MATMUL_CO_FUNCTIONS, MATMUL_I8_CO_FUNCTIONS

A, B, C, BIAS = 0x100000, 0x200000, 0x300000, 0x400000  # 16-byte aligned stand-ins, never dereferenced
F32, F16, BF16 = _native.DT_FLOAT32, _native.DT_FLOAT16, _native.DT_BFLOAT16
ES = {F32: 4, F16: 2, BF16: 2}
# TileArgs: a, b, c, vec, lda, ldb, ldc, M, N, K, tiles_m, tiles_n, out, act, alpha, trunc19, reserved
TILE_ARGS = struct.Struct("<QQQQqqqiiiiiiifii")


def lib():
    return _native.load_library()


def mm(fn, in_dt, out_dt, M, N, K, lda, ldb, ldc, a=A, act=0, alpha=0.0, bias=0):
    p = _native.LaunchPlan()
    return getattr(lib(), fn)(in_dt, out_dt, a, B, C, bias, M, N, K, lda, ldb, ldc, act, alpha, ctypes.byref(p)), p


def tile_of(name):
    bm, bn = re.search(r"(\d+)x(\d+)(?:k2)?$", name).groups()
    return int(bm), int(bn)


def check_tile(p, a, M, N, K, lda, ldb, ldc, es, offset):
    bm, bn = tile_of(p.kernel.decode())
    args = TILE_ARGS.unpack(p.blob())
    assert p.args_size == TILE_ARGS.size and args[0] == a and args[4:10] == (lda, ldb, ldc, M, N, K)
    tm, tn = -(-M // bm), -(-N // bn)
    assert args[10:12] == (tm, tn) and p.grid == tm * tn and p.grid * p.block < 2 ** 32
    aligned = offset % 16 == 0 and all(v * es % 16 == 0 for v in (lda, ldb, N, K))
    small = 256 * lda * es + K * es < 2 ** 31 - 2 ** 20 and 128 * ldb * es < 2 ** 31 - 2 ** 20
    assert ("_any_" not in p.kernel.decode()) == (aligned and small)


@settings(max_examples=600, deadline=None)
@given(in_dt=st.sampled_from([F32, F16, BF16]), out_dt=st.sampled_from([F32, F16, BF16]), M=st.integers(0, 20000),
       N=st.integers(0, 20000), K=st.integers(0, 20000), unit=st.sampled_from([1, 8, 256]), pad=st.integers(0, 64),
       a_off=st.sampled_from([0, 2, 16]))
def test_matmul_dispatch_properties(in_dt, out_dt, M, N, K, unit, pad, a_off):
    M, N, K = (v // unit * unit for v in (M, N, K))
    args = (in_dt, out_dt, M, N, K, K + pad, N, N)
    rc, p = mm("asc_matmul_dispatch", *args, a=A + a_off)
    rc0, p0 = mm("asc_matmul_plan", *args, a=A + a_off)
    assert rc == rc0
    if rc != 0 or M == 0 or N == 0:
        assert p.grid == 0
        return
    name = p.kernel.decode()
    assert name in MATMUL_CO_FUNCTIONS
    if "_tile_" not in name:  # the plan's own kernel, argument for argument
        assert (name, p.grid, p.block, p.blob()) == (p0.kernel.decode(), p0.grid, p0.block, p0.blob())
        assert K == 0 or "_fast_" in name or "f32_mfma" in name
        return
    assert K > 0 and f"_tile_{({F32: 'f32', F16: 'f16', BF16: 'bf16'}[in_dt])}_" in name
    check_tile(p, A + a_off, M, N, K, K + pad, N, N, ES[in_dt], a_off)
    assert TILE_ARGS.unpack(p.blob())[12] == {F32: 0, F16: 1, BF16: 2}[out_dt]


@settings(max_examples=400, deadline=None)
@given(M=st.integers(0, 30000), N=st.integers(0, 30000), K=st.integers(0, 1 << 17), unit=st.sampled_from([1, 16, 256]),
       dequant=st.booleans(), a_off=st.sampled_from([0, 1, 16]))
def test_int8_dispatch_properties(M, N, K, unit, dequant, a_off):
    M, N, K = (v // unit * unit for v in (M, N, K))
    p, p0 = _native.LaunchPlan(), _native.LaunchPlan()
    args = (A + a_off, B, BIAS, C, M, N, K, int(dequant), 1)
    assert lib().asc_matmul_i8_dispatch(*args, ctypes.byref(p)) == 0
    assert lib().asc_matmul_i8_plan(*args, ctypes.byref(p0)) == 0
    if M == 0 or N == 0:
        assert p.grid == 0
        return
    name = p.kernel.decode()
    assert name in MATMUL_I8_CO_FUNCTIONS
    if "_tile_" not in name:
        assert (name, p.grid, p.block, p.blob()) == (p0.kernel.decode(), p0.grid, p0.block, p0.blob())
        assert K == 0 or "_fast_" in name
        return
    check_tile(p, A + a_off, M, N, K, K, N, N, 1, a_off)
    out = TILE_ARGS.unpack(p.blob())
    assert (out[3], out[12], out[15]) == ((BIAS, 1, 1) if dequant else (0, 3, 0))


def test_dispatch_errors_match_the_plans():
    for args in ((F16, F16, 0, 0, 0, 0, -1, 8, 8, 8, 8, 8, 0, 0.0), (F16, F16, A, B, C, 0, 8, 8, 8, 4, 8, 8, 0, 0.0),
                 (F16, F16, 0, 0, C, 0, 8, 8, 8, 8, 8, 8, 0, 0.0), (3, F16, A, B, C, 0, 8, 8, 8, 8, 8, 8, 0, 0.0),
                 (F16, F16, A, B, C, 0, 8, 8, 8, 8, 8, 8, 3, 0.0),
                 (F16, F16, A, B, C, 0, 1 << 29, 1 << 29, 32, 32, 1 << 29, 1 << 29, 0, 0.0)):
        p = _native.LaunchPlan()
        assert lib().asc_matmul_dispatch(*args, ctypes.byref(p)) == lib().asc_matmul_plan(*args, ctypes.byref(p)) != 0
    p = _native.LaunchPlan()
    assert lib().asc_matmul_i8_dispatch(A, B, 0, C, 8, 8, 8, 1, 0, ctypes.byref(p)) == _native.ERR_INVALID_ARG
    assert lib().asc_matmul_i8_dispatch(A, B, 0, C, 8, 8, (1 << 17) + 1, 0, 0, ctypes.byref(p)) == \
        _native.ERR_UNSUPPORTED


def test_every_tile_kernel_is_reached():
    rng = random.Random(5)
    seen = set()
    for _ in range(6000):
        M, N, K = (int(2 ** rng.uniform(0, 13.5)) for _ in range(3))
        if rng.random() < 0.7:
            N, K = max(16, N // 16 * 16), max(16, K // 16 * 16)
        for dt in (F32, F16, BF16):
            seen.add(mm("asc_matmul_dispatch", dt, F32, M, N, K, K, N, N)[1].kernel.decode())
        p = _native.LaunchPlan()
        assert lib().asc_matmul_i8_dispatch(A, B, BIAS, C, M, N, K, 1, 0, ctypes.byref(p)) == 0
        seen.add(p.kernel.decode())
    assert {n for n in MATMUL_CO_FUNCTIONS + MATMUL_I8_CO_FUNCTIONS if "_tile_" in n} <= seen


def test_short_f32_products_take_blocks():
    # on both sides of each line: K, the number of blocks, the alignment, a few rows
    def name(M, N, K, a=A):
        rc, p = mm("asc_matmul_dispatch", F32, F32, M, N, K, K, N, N, a=a)
        assert rc == 0
        return p.kernel.decode()

    blocks = "asc2_mm_f32_mfma_f32"
    for M, N, K in ((1, 64, 4), (16, 16, 16), (64, 64, 64), (256, 256, 64), (512, 512, 16), (1, 4096, 256),
                    (260, 261, 57), (113, 1390, 137), (1, 11007, 101), (300, 301, 100)):
        assert name(M, N, K) == blocks, (M, N, K)
    for M, N, K in ((64, 64, 256), (256, 256, 256), (1, 4096, 1024), (1024, 1024, 64), (2048, 2048, 16),
                    (260, 261, 321), (1001, 1003, 101), (2049, 2049, 3)):
        assert name(M, N, K) != blocks, (M, N, K)
    assert name(64, 64, 256, a=A + 4) == blocks  # unaligned, up to 256 blocks: whatever K


def test_tile_aligned_products_keep_their_loop():
    # from 129 to 256 tiles of 256x256 every other tile is the slower one; above, 192x128 is where it
    # fills about as many rounds
    def names(M, N, K):
        rc, p = mm("asc_matmul_dispatch", BF16, BF16, M, N, K, K, N, N)
        q = _native.LaunchPlan()
        assert rc == 0 and lib().asc_matmul_i8_dispatch(A, B, BIAS, C, M, N, K, 1, 0, ctypes.byref(q)) == 0
        return p.kernel.decode(), q.kernel.decode()

    for tm in range(1, 40):
        for tn in (1, 3, 8, 12, 16, 24, 43):
            for K in (64, 1024, 4096, 11008, 1 << 16):
                if 128 < tm * tn <= 256:
                    assert all("_fast_" in n for n in names(256 * tm, 256 * tn, K)), (tm, tn, K)
    for M, N, K in ((6144, 4096, 11008), (5632, 4096, 11008), (6144, 6144, 4096), (2048, 11008, 11008)):
        assert not any("192x128" in n for n in names(M, N, K)), (M, N, K)
    assert all("192x128" in n for n in names(1536, 4096, 4096))  # one round of 192x128
    assert all("192x128" in n for n in names(4608, 4096, 11008))  # three full rounds, the loop's two with 32 tiles
    assert all("192x128" in n for n in names(3000, 4096, 4096))  # no multiple of 256: the loop cannot take it


@settings(max_examples=1500, deadline=None)
@given(in_dt=st.sampled_from([F32, F16, BF16]), out_dt=st.sampled_from([F32, F16, BF16]), M=st.integers(1, 12),
       N=st.integers(1, 24), K=st.integers(1, 24), pad=st.integers(0, 40), shift=st.integers(-130, 130),
       other=st.sampled_from("ab"))
def test_products_in_place_keep_the_plans_kernel(in_dt, out_dt, M, N, K, pad, shift, other):
    # C and an operand with one row pitch, C's rows moved by less than that: every byte of both, one
    # by one.  Tiles take the product if and only if it shares none, or is fp32 (in 16x16 blocks or
    # small tiles, of which one holds up to 16 columns as well).
    es, oes = ES[in_dt], ES[out_dt]
    pitch = (max(K * es, N * es, N * oes) + pad) // 4 * 4 + 4
    at = A + shift % pitch // oes * oes * (1 if shift >= 0 else -1)
    a, b = (A, 0x4000000) if other == "a" else (0x4000000, A)
    lda, ldb = (pitch // es, N) if other == "a" else (K, pitch // es)
    rows, cols = (M, K) if other == "a" else (K, N)
    p = _native.LaunchPlan()
    assert lib().asc_matmul_dispatch(in_dt, out_dt, a, b, at, 0, M, N, K, lda, ldb, pitch // oes, 0, 0.0,
                                     ctypes.byref(p)) == 0
    taken = {A + r * pitch + i for r in range(rows) for i in range(cols * es)}
    shared = any(at + r * pitch + i in taken for r in range(M) for i in range(N * oes))
    if in_dt != F32 and shared:
        assert "_tile_" not in p.kernel.decode()
    elif in_dt != F32 and M > 1 and rows > 1:  # (with a single row a neighbour's does not exist)
        assert "_tile_" in p.kernel.decode()


def test_in_place_beyond_one_workgroup_or_a_pitch_is_no_concern():
    def tile(M, N, K, c, other_b=B, ldc=None):
        p = _native.LaunchPlan()
        assert lib().asc_matmul_dispatch(BF16, BF16, A, other_b, c, 0, M, N, K, K, N, ldc or N, 0, 0.0,
                                         ctypes.byref(p)) == 0
        return "_tile_" in p.kernel.decode()

    assert not tile(1000, 256, 256, A) and tile(1000, 264, 264, A)  # more columns: never one workgroup's rows
    assert not tile(256, 256, 256, B) and tile(257, 256, 257, B)    # in place of B: one workgroup
    assert tile(1000, 64, 128, A)                                   # another pitch
    assert not tile(1000, 64, 128, A, ldc=128) and tile(1000, 64, 64, A + 128, ldc=128)
    for dequant, width in ((0, 4), (1, 2)):
        for at, shared in ((A, True), (A + 256, False), (A - 64 * width, False), (A + 100, True)):
            p = _native.LaunchPlan()
            assert lib().asc_matmul_i8_dispatch(A, B, BIAS, at, 300, 64, 64 * width, dequant, 0, ctypes.byref(p)) == 0
            assert ("_tile_" in p.kernel.decode()) == (not shared), (dequant, hex(at))
