"""SwiGLU gradients whose output just fits, and just exceeds, what is written with ordinary stores (128 MiB), against the same
kernel on pieces of 1000 rows (always ordinary stores): equal bit for bit.  The output's memory held NaN before."""
import pytest
import torch

import mindspeed_amd.ops as ops

pytestmark = pytest.mark.gpu

LIMIT = 128 << 20


def gradients(x, probs, gy):
    x, probs = x.detach().requires_grad_(True), probs.detach().requires_grad_(True)
    return torch.autograd.grad(ops.swiglu_with_probs(x, probs), (x, probs), gy)


# (13 columns: no 16-byte vectors)
@pytest.mark.parametrize("ffn,dtype", [(4096, torch.bfloat16), (4096, torch.float16), (2048, torch.float32), (13, torch.bfloat16)])
def test_equals_the_gradients_of_pieces(ffn, dtype):
    row = 2 * ffn * torch.empty(0, dtype=dtype).element_size()
    for rows in (LIMIT // row, LIMIT // row + 1):
        print(ffn, dtype, rows, flush=True)
        gen = torch.Generator(device="cuda").manual_seed(ffn)
        x = torch.randn(rows, 2 * ffn, generator=gen, device="cuda").to(dtype)
        gy = torch.randn(rows, ffn, generator=gen, device="cuda").to(dtype)
        probs = torch.rand(rows, generator=gen, device="cuda").to(dtype)
        step = 1000 if ffn > 100 else 1 << 19
        want = [gradients(x[r:r + step], probs[r:r + step], gy[r:r + step]) for r in range(0, rows, step)]
        held = [torch.full_like(x, float("nan")) for _ in range(3)]
        del held
        dx, dp = gradients(x, probs, gy)
        assert torch.equal(dx, torch.cat([a for a, _ in want])) and torch.equal(dp, torch.cat([b for _, b in want]))
