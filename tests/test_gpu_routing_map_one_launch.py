"""The routing-map permute that writes probabilities and token numbers beside the rows, and the unpermute gradient that
zeroes unmapped rows, against the separate kernels: moved bits and zeros, so everything is equal."""
import pytest
import torch

from mindspeed_amd.ops._kernels import K

pytestmark = pytest.mark.gpu

# tokens, experts, rows beyond the set entries, hidden, tokens' dtype, probabilities' dtype, drop-and-pad capacity:
# both kernels that rank the map (a power of two up to 16 experts; any), the sort behind them (drop-and-pad, more experts
# than a workgroup's lists hold), one token, rows that are no whole 16-byte vectors, unmapped rows
CASES = [
    (1, 8, 0, 64, torch.bfloat16, torch.float32, 0),
    (700, 8, 61, 256, torch.bfloat16, torch.bfloat16, 0),
    (513, 16, 0, 8, torch.float32, torch.float32, 0),
    (300, 2, 3, 72, torch.float16, torch.float16, 0),
    (333, 60, 1100, 192, torch.bfloat16, torch.float32, 0),
    (300, 6, 5, 70, torch.float32, torch.float32, 0),
    (1025, 12, 0, 33, torch.bfloat16, torch.float32, 0),
    (300, 900, 53, 32, torch.bfloat16, torch.bfloat16, 0),
    (128, 8, 0, 64, torch.bfloat16, torch.float32, 40),
]


@pytest.mark.parametrize("T,E,extra,H,dtype,pdtype,capacity", CASES)
@pytest.mark.parametrize("with_probs", [True, False])
def test_equals_the_separate_kernels(T, E, extra, H, dtype, pdtype, capacity, with_probs):
    gen = torch.Generator(device="cuda").manual_seed(T + E)
    rmap = torch.rand(T, E, generator=gen, device="cuda") < min(2.0 / E, 0.5)
    rows = E * capacity if capacity else int(rmap.sum()) + extra
    tokens = torch.randn(T, H, generator=gen, device="cuda").to(dtype)
    probs = torch.rand(T, E, generator=gen, device="cuda").to(pdtype) if with_probs else None
    pad = capacity > 0
    perm, rid, flat, _ = K.routing_map_permute(tokens, rmap, rows, pad, False)
    pp, ids = K.routing_map_probs(flat, probs, E)
    poison = torch.full((1 << 22,), float("nan"), device="cuda")
    del poison
    one = K.routing_map_permute_probs(tokens, rmap, probs, rows, pad)
    for a, b in zip(one, (perm, rid, flat, pp, ids)):
        assert torch.equal(a, b)

    gy = torch.randn(T, H, generator=gen, device="cuda").to(dtype)
    p = probs.to(dtype) if probs is not None and pdtype != torch.float32 else probs
    empty = perm if p is not None else perm.new_empty(0)
    g, gp = K.moe_token_unpermute_grad(empty, gy, rid, p, T, E, rows)
    K.zero_unmapped_rows(g, flat)
    poison = torch.full((1 << 22,), float("nan"), device="cuda")
    del poison
    g1, gp1 = K.moe_token_unpermute_grad(empty, gy, rid, p, T, E, rows, flat)
    assert torch.equal(g, g1) and torch.equal(gp, gp1)
    assert not torch.isnan(g1).any()
