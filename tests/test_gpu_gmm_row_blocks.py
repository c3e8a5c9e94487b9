"""A full-height tile that a group fills in part computes its rows in 32-row blocks, as many as it takes.  The same rows in groups
that fill their tiles run through all eight blocks; a row's sums are formed in the same order either way, so the results are equal
bit for bit."""
import pytest
import torch

from conftest import rel_l2
from mindspeed_amd.ops._kernels import K
from mindspeed_amd.ops.gmm import gmm_backward_raw, gmm_raw

pytestmark = pytest.mark.gpu

# one tile of rows per group, both edges of every number of blocks; by 12 column tiles they are 132, more than half a round of
# compute units, so that the launch does not divide them
ROWS = [129, 144, 145, 160, 161, 176, 192, 193, 224, 225, 255]
N = 12 * 256


def _rows(k, dtype):
    """The groups' rows, packed and each filled up to 256, and which of the latter they are."""
    gen = torch.Generator(device="cuda").manual_seed(k)
    full = torch.randn(256 * len(ROWS), k, generator=gen, device="cuda").to(dtype)
    own = torch.cat([torch.arange(r, device="cuda") + 256 * g for g, r in enumerate(ROWS)])
    counts = torch.tensor(ROWS, device="cuda")
    return full, own, counts, torch.full_like(counts, 256)


def _weight(k, n, dtype):
    gen = torch.Generator(device="cuda").manual_seed(n)
    return (0.1 * torch.randn(len(ROWS), k, n, generator=gen, device="cuda")).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k,n", [(8, N), (64, N - 8), (72, N), (128, N - 120), (328, N)])
def test_equals_tiles_that_are_full(k, n, dtype):
    full, own, counts, whole = _rows(k, dtype)
    w = _weight(k, n, dtype)
    x = full[own].contiguous()
    along_n = w.transpose(1, 2).contiguous().transpose(1, 2)
    for weight in (w, along_n):
        y = torch.full((x.size(0) + 3, n), float("nan"), dtype=dtype, device="cuda")
        gmm_raw(x, weight, counts, 0, 1, out=y[:-3])
        assert torch.equal(y[:-3], gmm_raw(full, weight, whole, 0, 1)[own])
        assert bool(y[-3:].isnan().all())
        expect = torch.cat([a.double() @ b.double() for a, b in zip(x.split(ROWS), w)])
        assert rel_l2(y[:-3], expect) <= (4e-3 if dtype == torch.bfloat16 else 5e-4)      # one rounding: 2^-9, 2^-12 at most


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k,ffn", [(72, N // 2), (128, N // 2 - 8), (64, N // 2 - 56), (200, N // 2 - 72)])
def test_activation_in_the_epilogue(k, ffn, dtype):
    full, own, counts, whole = _rows(k, dtype)
    w = _weight(k, 2 * ffn, dtype)
    x = full[own].contiguous()
    for probs in (None, torch.rand(full.size(0), device="cuda"), torch.rand(full.size(0), device="cuda").to(dtype)):
        mine = None if probs is None else probs[own].contiguous()
        fc1, act = K.gmm_swiglu(x, w, counts, 1, mine, True)
        assert torch.equal(fc1, gmm_raw(x, w, counts, 0, 1))
        assert torch.equal(act, K.swiglu(fc1, mine))                       # the kernel of its own
        assert torch.equal(act, K.gmm_swiglu(x, w, counts, 1, mine, False)[1])
        fc1_full, act_full = K.gmm_swiglu(full, w, whole, 1, probs, True)
        assert torch.equal(fc1, fc1_full[own]) and torch.equal(act, act_full[own])


@pytest.mark.parametrize("accumulate", [False, True])
def test_gradient_of_the_rows_in_one_launch_with_the_weight(accumulate):
    k, dtype = 12 * 256, torch.bfloat16                 # (dX has the columns that the forward sums over)
    full, own, counts, whole = _rows(136, dtype)        # the incoming gradient
    w = _weight(k, 136, dtype)
    x = torch.randn(full.size(0), k, device="cuda").to(dtype)
    out = torch.float32 if accumulate else dtype
    dw, dw_apart = torch.zeros(len(ROWS), k, 136, dtype=out, device="cuda"), torch.zeros(len(ROWS), k, 136, dtype=out, device="cuda")
    dx = gmm_backward_raw(full[own].contiguous(), x[own].contiguous(), w, counts, 1, dw, accumulate)
    assert torch.equal(dx, gmm_raw(full, w.transpose(1, 2), whole, 0, 1)[own])
    gmm_raw(x[own].contiguous().t(), full[own].contiguous(), counts, 2, 1, out=dw_apart, accumulate=accumulate)
    assert torch.equal(dw, dw_apart)
