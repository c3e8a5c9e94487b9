"""The sigmoid of the 16-bit SwiGLU kernels where exp(-x) comes near the largest 32-bit value or vanishes beside 1: the values that
test_gpu_swiglu_sigmoid.py leaves out.  exp(-x) is finite in 32 bits down to x = -88.72 and sigmoid(x) a subnormal from -87.34 on,
but x * sigmoid(x) is a normal bfloat16 there."""
import pytest
import torch

from mindspeed_amd.ops._kernels import K

pytestmark = pytest.mark.gpu

FFN = 128


def _gates(dtype):
    """All finite values outside (-80, 80), in rows of FFN (the last one filled up with zeros)."""
    x = torch.arange(-2 ** 15, 2 ** 15, dtype=torch.int32).to(torch.int16).view(dtype)
    x = x[x.isfinite() & (x.double().abs() >= 80)]
    return torch.cat([x, x.new_zeros(-x.numel() % FFN)]).view(-1, FFN).to("cuda")


def _check(gate, act, grad):
    x, dtype = gate.double(), gate.dtype
    sig = torch.sigmoid(x)
    step = torch.finfo(dtype).eps / 2                    # half a unit in the last place, of values that are not denormal
    slack = 4e-7 * (1 + x.abs())                         # exp(-x) in 32 bits is off by |x| 2^-24 and a few units more
    tiny = torch.finfo(dtype).smallest_normal * step     # half the smallest denormal
    high, low, over = x >= 80, (x <= -80) & (x > -88.7), x < -88.75
    if act is not None:
        assert bool((act.double() == x)[high].all())
        err = (act.double() - x * sig).abs()
        assert bool((err <= (step + 1.01 * slack) * (x * sig).abs() + tiny)[low].all())
        assert bool((act == 0)[over].all())              # exp overflows: zero, as the division gives
    if grad is not None:
        expect = sig * (1 + x * (1 - sig))
        assert bool((grad == 1)[high].all())
        err = (grad.double() - expect).abs()
        assert bool((err <= step * expect.abs() + 1.01 * slack * (1 + x.abs()) * sig + tiny)[low].all())
        assert bool((grad == 0)[over].all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_kernels_of_their_own(dtype):
    gate = _gates(dtype)
    one = torch.ones_like(gate)
    rows = torch.cat([gate, one], dim=1)
    d = K.swiglu_grad(one, rows, None)[0]
    _check(gate, K.swiglu(rows, None), d[:, :FFN])


@pytest.mark.parametrize("per_group", [40, 256])         # small tiles and full ones
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_epilogues_of_the_grouped_matmul(dtype, per_group):
    """The first matmul's output is the gate itself beside ones: x = (gate values, 1), weight = (identity, 0; 0, ones)."""
    gate = _gates(dtype)
    m, ffn = gate.size(0), FFN
    x = torch.cat([gate, torch.ones(m, 8, dtype=dtype, device="cuda")], dim=1)
    groups = (m + per_group - 1) // per_group
    counts = torch.full((groups,), per_group, device="cuda")
    counts[-1] = m - per_group * (groups - 1)
    w = torch.zeros(groups, ffn + 8, 2 * ffn, dtype=dtype, device="cuda")
    w[:, :ffn, :ffn] = torch.eye(ffn, dtype=dtype, device="cuda")
    w[:, ffn, ffn:] = 1
    fc1, act = K.gmm_swiglu(x, w, counts, 1, None, True)
    assert torch.equal(fc1, torch.cat([gate, torch.ones_like(gate)], dim=1))
    dy = torch.zeros(m, 8, dtype=dtype, device="cuda")
    dy[:, 0] = 1
    w2 = torch.zeros(groups, ffn, 8, dtype=dtype, device="cuda")
    w2[:, :, 0] = 1                                      # d(activation) = 1
    d, _ = K.gmm_swiglu_grad(dy, w2, fc1, None, counts, 1)
    _check(gate, act, d[:, :ffn])
