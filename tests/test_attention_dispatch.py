"""asc_flash_attention_dispatch without a GPU (non-causal: a causal launch asks the device for
its CUs): asc_flash_attention_plan's launch, or the kernel that splits the keys with a
workgroup per 32 queries, the same arguments otherwise and the same errors."""
import ctypes
import random
import struct

from pyasc_amd import _native
from pyasc_amd.launchers import ATTENTION_CODE_OBJECT

Q, K, V, O, LSE = 0x10000, 0x20000, 0x30000, 0x40000, 0x50000  # stand-ins, never dereferenced
# FaArgs: q, k, v, o, lse, heads_total, seq, n_qblocks, head_group, scale_log2, causal
FA_ARGS = struct.Struct("<QQQQQqiiifi4x")


def both(*args):
    lib = _native.load_library()
    p, d = _native.LaunchPlan(), _native.LaunchPlan()
    return (lib.asc_flash_attention_plan(*args, ctypes.byref(p)), p,
            lib.asc_flash_attention_dispatch(*args, ctypes.byref(d)), d)


def test_launch_against_the_plan():
    rng = random.Random(7)
    seen = set()
    for _ in range(4000):
        b, h, s = rng.randint(1, 8), int(2 ** rng.uniform(0, 8)), int(2 ** rng.uniform(0, 16))
        dim = rng.choice((64, 128))
        rc, p, drc, d = both(Q, K, V, O, LSE, b, h, s, dim, 0.125, 0)
        assert rc == drc == 0
        name = d.kernel.decode()
        seen.add(name)
        pa, da = FA_ARGS.unpack(p.blob()), FA_ARGS.unpack(d.blob())
        if name.endswith("_split"):
            assert name == p.kernel.decode() + "_split" and d.block == 256
            assert da[7] == -(-s // 32) and d.grid == b * h * da[7]
            assert pa[:7] + pa[8:] == da[:7] + da[8:]
        else:
            assert (name, d.grid, d.block, da) == (p.kernel.decode(), p.grid, p.block, pa)
    assert seen == set(ATTENTION_CODE_OBJECT.functions)


def test_errors_are_the_plans():
    for args in ((Q, K, V, O, 0, 1, 1, 64, 96, 0.1, 0), (Q, K, V, O, 0, 1, 1, 64, 64, -1.0, 0),
                 (Q + 8, K, V, O, 0, 1, 1, 64, 64, 0.1, 0), (0, K, V, O, 0, 1, 1, 64, 64, 0.1, 0),
                 (Q, K, V, O, 0, -1, 1, 64, 64, 0.1, 0), (Q, K, V, O, 0, 1, 1, 1 << 30, 64, 0.1, 0),
                 (Q, K, V, O, 0, 1 << 20, 1 << 20, 64, 64, 0.1, 0)):
        rc, _, drc, _ = both(*args)
        assert rc == drc != 0
    rc, p, drc, d = both(0, 0, 0, 0, 0, 0, 8, 64, 64, 0.1, 0)
    assert rc == drc == 0 and p.grid == d.grid == 0
