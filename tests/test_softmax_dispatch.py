"""asc_softmax_dispatch without a GPU: the launch the softmax entries make covers the plan's
rows with the plan's arguments, by a kernel that holds rows of that length, and fails exactly
where the plan fails.  Over many shapes the choice reaches every kernel that only it names."""
import ctypes
import random

from pyasc_amd import _native
from pyasc_amd.launchers import SOFTMAX_CO_FUNCTIONS, SOFTMAX_DISPATCH_FUNCTIONS

F32, F16 = _native.DT_FLOAT32, _native.DT_FLOAT16
X, OUT = 0x10000, 0x20000  # stand-ins, never dereferenced


def both(*args):
    lib = _native.load_library()
    p, d = _native.SoftmaxPlan(), _native.SoftmaxPlan()
    return (lib.asc_softmax_plan(*args, ctypes.byref(p)), p), (lib.asc_softmax_dispatch(*args, ctypes.byref(d)), d)


def test_launch_against_the_plan():
    rng = random.Random(4)
    seen = set()
    for _ in range(20000):
        dtype = rng.choice((F32, F16))
        rows, cols = int(2 ** rng.uniform(0, 23)), int(2 ** rng.uniform(0, 17.5))
        fused = rng.random() < 0.3
        size = int(2 ** rng.uniform(0, 10)) if fused else rng.choice((cols, cols, max(1, cols // 2), cols + 3))
        grid = rng.choice((0, 1, 16, 500))
        (rc, p), (drc, d) = both(dtype, fused, X + 4 * rng.randrange(4), OUT, rows, cols, size, grid)
        assert rc == drc
        if rc:
            continue
        assert (p.grid == 0) == (d.grid == 0)
        assert (p.rows, p.stride, p.len, p.flag) == (d.rows, d.stride, d.len, d.flag)
        if not d.grid:
            continue
        name = d.kernel.decode()
        seen.add(name)
        if name == "asc2_softmax_short_f32":
            assert dtype == F32 and d.len <= 512 and d.block == 256 and d.grid == -(-d.rows // 16)
        elif name == "asc2_softmax_wide_f32":
            assert dtype == F32 and d.block == 1024 and d.grid == d.rows and d.rows * 1024 < 2 ** 32
        elif name == "asc2_softmax_wide_f16":
            assert dtype == F16 and d.block == 1024 and d.grid == min(d.rows, 65536)
        else:
            assert (name, d.block) == (p.kernel.decode(), p.block)
            assert d.grid <= p.grid if name == "asc2_softmax_f16" else d.grid == p.grid
    assert seen == set(SOFTMAX_DISPATCH_FUNCTIONS)
    assert set(SOFTMAX_CO_FUNCTIONS) < seen


def test_errors_are_the_plans():
    for args in ((F32, 0, 0, OUT, 4, 4, 4, 1), (9, 0, X, OUT, 4, 4, 4, 1), (F16, 0, X, OUT, -1, 4, 4, 1),
                 (F32, 1, X, OUT, 4, 0, 4, 1), (F16, 1, X, OUT, 4, 4, 0, 1)):
        (rc, _), (drc, _) = both(*args)
        assert rc == drc
    assert _native.load_library().asc_softmax_dispatch(F32, 0, X, OUT, 4, 4, 4, 1, None) == _native.load_library() \
        .asc_softmax_plan(F32, 0, X, OUT, 4, 4, 4, 1, None) != 0
