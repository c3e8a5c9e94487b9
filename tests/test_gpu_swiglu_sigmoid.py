"""The sigmoid of the 16-bit SwiGLU kernels (a reciprocal and one Newton step) over every value of the types."""
import pytest
import torch

from mindspeed_amd.ops._kernels import K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_sigmoid_over_every_16_bit_value(dtype):
    """silu and its derivative of all finite values, and what the division gives at infinities and NaN."""
    bits = torch.arange(-2 ** 15, 2 ** 15, dtype=torch.int32).to(torch.int16)
    x = bits.view(dtype).to("cuda")
    one = torch.ones_like(x)
    rows = torch.cat([x.view(64, -1), one.view(64, -1)], dim=1).contiguous()
    act = K.swiglu(rows, None).view(-1)
    grad = K.swiglu_grad(one.view(64, -1).contiguous(), rows, None)[0][:, :1024].reshape(-1)
    x64 = x.double()
    sig = torch.sigmoid(x64)
    step = torch.finfo(dtype).eps / 2                    # half a unit in the last place, of values that are not denormal
    # exp(-x) in 32 bits is off by |x| 2^-24 and a few units more, 1 - sigmoid(x) by 2^-24
    slack = 4e-7 * (1 + x64.abs())
    for got, expect, off in ((act, x64 * sig, slack * (x64 * sig).abs()), (grad, sig * (1 + x64 * (1 - sig)), slack * (1 + x64.abs()) * sig)):
        finite = x64.isfinite() & (x64.abs() < 80) & (expect.abs() < torch.finfo(dtype).max)
        err = (got.double() - expect).abs()
        bound = step * expect.abs() + 1.01 * off + torch.finfo(dtype).smallest_normal * step
        assert bool((err <= bound)[finite].all())
    assert bool(act[x.isnan()].isnan().all())
    assert bool((act[x64 == float("inf")] == float("inf")).all()) and bool(act[x64 == float("-inf")].isnan().all())
    low = x64.isfinite() & (x64 < -104)                  # exp overflows: zero, as the division gives
    assert bool((act[low] == 0).all())
