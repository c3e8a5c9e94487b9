"""A Recorder that wants the launches of an unrecorded backward pass sees the two gradients of a grouped matmul as one call, by
default as two; the results are the unrecorded ones."""
import pytest
import torch

from mindspeed_amd import flop_counter
from mindspeed_amd.dispatcher import dispatch_mlp_combine

pytestmark = pytest.mark.gpu

GRADIENTS = {"gmm_dx_and_dw", "gmm_dx", "gmm_dw"}


@pytest.mark.parametrize("gemm_fusion", [False, True])
@pytest.mark.parametrize("pairs", [False, True])
def test_gradients_of_a_matmul(pairs, gemm_fusion):
    gen = torch.Generator(device="cuda").manual_seed(0)
    x, w1, w2 = (torch.randn(*s, generator=gen, device="cuda").bfloat16() for s in ((40, 64), (4, 64, 48), (4, 24, 64)))
    index = torch.arange(80, device="cuda").view(40, 2) % 4
    probs = torch.rand(40, 2, generator=gen, device="cuda").bfloat16()

    def layer():
        leaves = [t.detach().requires_grad_(True) for t in (x, w1, w2)]
        for w in leaves[1:]:
            w.main_grad = torch.zeros(w.shape, device="cuda")
        y = dispatch_mlp_combine(leaves[0], index, probs, leaves[1:], gemm_fusion=gemm_fusion)
        if gemm_fusion:
            return [y.detach(), *torch.autograd.grad(y, leaves[:1], torch.ones_like(y)), *(w.main_grad for w in leaves[1:])]
        return [y.detach(), *torch.autograd.grad(y, leaves, torch.ones_like(y))]

    plain = layer()
    with flop_counter.record(timing=False, pairs=pairs) as rec:
        got = layer()
    assert all(torch.equal(a, b) for a, b in zip(plain, got))
    names = [c[0] for c in rec.calls if c[0] in GRADIENTS]
    assert sorted(names) == (["gmm_dx_and_dw"] * 2 if pairs else ["gmm_dw"] * 2 + ["gmm_dx"] * 2)
    flops = sum(c[1] for c in rec.calls if c[0] in GRADIENTS)
    assert flops == 2 * (flop_counter.gmm_flops(80, 64, 48) + flop_counter.gmm_flops(80, 24, 64))
