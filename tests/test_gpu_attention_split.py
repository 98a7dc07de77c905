"""Attention whose keys are split over waves, and the kernel without the split, on the same
inputs at the edges of query blocks, key tiles and the rounds of four tiles: each against fp64
within the rounding of its probabilities and output to bf16, a late key that moves the
reference point of one wave only, and queries whose waves have no keys."""
import pytest
import torch

from pyasc_amd import kernels
from pyasc_amd.asc.runtime import module
from pyasc_amd.launchers import ATTENTION_CODE_OBJECT

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def functions(device):
    return module.load(ATTENTION_CODE_OBJECT, str(ATTENTION_CODE_OBJECT.path)).functions


def _check(q, k, v, o, lse, scale, causal):
    S, D = q.shape[2:]
    qd, kt, vd = q.double(), k.double().transpose(-1, -2).contiguous(), v.double()
    s = (qd @ kt) * scale
    if causal:
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    p = torch.softmax(s, dim=-1)
    ref, mag = p @ vd, p @ vd.abs()
    # fp32: D products per score and the FMA before exp2, S terms per sum; bf16 (eight
    # significant bits, so rounding moves a value by up to 2^-8 of it): the probabilities, and
    # the result
    eps = (D + 4) * 2.0 ** -23 * float((qd.abs() @ kt.abs()).max()) * scale + (S + 16) * 2.0 ** -22
    bound = mag * (2.0 ** -8 + eps)
    bound = bound + 2.0 ** -8 * (ref.abs() + bound) + 2.0 ** -120
    assert ((o.double() - ref).abs() <= bound).all()
    want = torch.logsumexp(s, dim=-1)
    assert ((lse.double() - want).abs() <= eps + 2.0 ** -22 * (want.abs() + 1)).all()


def _run(functions, q, k, v, causal, split):
    scale = q.shape[3] ** -0.5
    for dispatched in (True, False):
        o, lse = torch.full_like(q, 7.0), torch.full(q.shape[:3], 7.0, device=q.device)
        plan = (kernels.flash_attention_dispatch if dispatched else kernels.flash_attention_plan)(
            q, k, v, o, scale, causal, lse)
        assert plan.kernel.decode().endswith("_split") == (dispatched and split)
        if dispatched:
            kernels.flash_attention_fwd(q, k, v, o, scale, causal, lse=lse)
        else:
            module.launch_plan(functions, plan, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        _check(q, k, v, o, lse, scale, causal)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,S", [(1, 1, 1), (1, 3, 31), (2, 8, 32), (1, 1, 33), (3, 1, 64), (1, 2, 65), (1, 8, 127),
                                   (1, 1, 129), (1, 5, 255), (2, 4, 257), (1, 1, 289), (1, 2, 513), (1, 16, 777),
                                   (1, 1, 4097)])
def test_edges(device, functions, B, H, S, D, causal):
    g = torch.Generator(device=device).manual_seed(S + D)
    q, k, v = (torch.randn((B, H, S, D), generator=g, device=device).bfloat16() for _ in range(3))
    _run(functions, q, k, v, causal, split=True)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("late", [3, 70, 200, 390, 600, 999])
def test_a_late_key_far_above_the_rest(device, functions, D, late):
    g = torch.Generator(device=device).manual_seed(late)
    q, k, v = (torch.randn((1, 2, 1000, D), generator=g, device=device).bfloat16() for _ in range(3))
    q[..., 0] = 8.0
    k[:, :, late, 0] = 8.0 * D ** 0.5 / 4
    _run(functions, q, k, v, False, split=True)
    _run(functions, q, k, v, True, split=True)


@pytest.mark.parametrize("D", [64, 128])
def test_many_heads_are_not_split(device, functions, D):
    g = torch.Generator(device=device).manual_seed(D)
    q, k, v = (torch.randn((2, 64, 500, D), generator=g, device=device).bfloat16() for _ in range(3))
    _run(functions, q, k, v, True, split=False)
