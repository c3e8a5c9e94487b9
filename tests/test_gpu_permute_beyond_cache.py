"""Permutes whose tokens and rows together just fit, and just exceed, what is written with ordinary stores (320 MiB): every
kernel that scatters rows, 16-byte and narrower vectors.  Rows are copies, so everything is equal; the output's memory held NaN
before."""
import pytest
import torch

import mindspeed_amd.ops as ops
from mindspeed_amd.ops._kernels import K

pytestmark = pytest.mark.gpu

LIMIT = 320 << 20
# tokens, top-k, experts, hidden sizes at and beyond the limit (16-bit rows)
CASES = {
    "counted_by_the_movers": (2048, 8, 8, (9096, 9104)),
    "counted_by_the_movers_16": (2048, 8, 12, (9096, 9104)),
    "counters_per_expert": (2048, 8, 64, (9096, 9104)),
    "behind_a_histogram": (4096, 8, 64, (4544, 4552, 4553)),
}


def poison(like):
    held = [torch.full_like(like, float("nan")) for _ in range(3)]
    del held


@pytest.mark.parametrize("name", CASES)
def test_rows_are_copies(name):
    T, k, E, hiddens = CASES[name]
    gen = torch.Generator(device="cuda").manual_seed(T + E)
    idx = torch.topk(torch.rand(T, E, generator=gen, device="cuda"), k, dim=-1)[1]
    assert [(T + T * k) * H * 2 <= LIMIT for H in hiddens] == [True] + [False] * (len(hiddens) - 1)
    for H in hiddens:
        print(name, H, flush=True)
        tokens = torch.randn(T, H, generator=gen, device="cuda").bfloat16()
        want = tokens.repeat_interleave(k, 0)[torch.argsort(idx.reshape(-1), stable=True)]
        poison(want)
        perm, _, _, _ = ops.moe_token_permute_with_aux(tokens, idx, num_experts=E)
        assert torch.equal(perm, want)


@pytest.mark.parametrize("E", [8, 60])
def test_rows_of_a_routing_map_are_copies(E):
    T, k = 2048, 8
    gen = torch.Generator(device="cuda").manual_seed(E)
    idx = torch.topk(torch.rand(T, E, generator=gen, device="cuda"), k, dim=-1)[1]
    rmap = torch.zeros(T, E, dtype=torch.bool, device="cuda").scatter_(1, idx, True)
    token_of_row = rmap.t().nonzero()[:, 1]
    for H in (9096, 9104):
        print(E, H, flush=True)
        tokens = torch.randn(T, H, generator=gen, device="cuda").bfloat16()
        want = tokens[token_of_row]
        poison(want)
        perm = K.routing_map_permute(tokens, rmap, T * k, False, False)[0]
        assert torch.equal(perm, want)
