"""Row blocks of a full-height tile that a group fills in part, and shared last tiles, with the outputs that test_gpu_gmm_row_blocks.py
leaves out: fp32, `+=` into fp32, and the SwiGLU backward in the epilogue.  The same rows in groups that fill their tiles run through
all eight blocks; a row's sums are formed in the same order either way, so the results are equal bit for bit."""
import pytest
import torch

from mindspeed_amd.ops._kernels import K
from mindspeed_amd.ops.gmm import gmm_raw

pytestmark = pytest.mark.gpu

# both edges of every number of blocks; two tiles that share their rows (at least 97 and 160, at most 192 each)
ROWS = [129, 160, 161, 192, 193, 224, 225, 255, 256, 257, 320, 321, 384]
N = 8 * 256           # 17 row tiles: 136 tiles, more than half a round, so that the launch does not divide them


def _inputs(k, dtype):
    gen = torch.Generator(device="cuda").manual_seed(k)
    whole = [(r + 255) // 256 * 256 for r in ROWS]
    full = torch.randn(sum(whole), k, generator=gen, device="cuda").to(dtype)
    first = torch.tensor([0] + whole).cumsum(0).tolist()
    own = torch.cat([torch.arange(r, device="cuda") + b for r, b in zip(ROWS, first)])
    return full, own, torch.tensor(ROWS, device="cuda"), torch.tensor(whole, device="cuda"), gen


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k,n", [(8, N), (72, N - 8), (328, N - 120)])
def test_fp32_output(k, n, dtype):
    full, own, counts, whole, gen = _inputs(k, dtype)
    x = full[own].contiguous()
    w = (0.1 * torch.randn(len(ROWS), k, n, generator=gen, device="cuda")).to(dtype)
    for weight in (w, w.transpose(1, 2).contiguous().transpose(1, 2)):
        expect = torch.empty(full.size(0), n, device="cuda")
        gmm_raw(full, weight, whole, 0, 1, out=expect)
        y = torch.full((x.size(0) + 3, n), float("nan"), device="cuda")
        gmm_raw(x, weight, counts, 0, 1, out=y[:-3])
        assert torch.equal(y[:-3], expect[own]) and bool(y[-3:].isnan().all())
        old = torch.randn(x.size(0), n, generator=gen, device="cuda")
        y[:-3] = old
        gmm_raw(x, weight, counts, 0, 1, out=y[:-3], accumulate=True)
        assert torch.equal(y[:-3], old + expect[own]) and bool(y[-3:].isnan().all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hidden,ffn", [(8, N), (72, N - 8), (328, N - 120)])
def test_swiglu_backward_in_the_epilogue(hidden, ffn, dtype):
    full, own, counts, whole, gen = _inputs(hidden, dtype)
    w2 = (0.1 * torch.randn(len(ROWS), ffn, hidden, generator=gen, device="cuda")).to(dtype)
    fc1 = torch.randn(full.size(0), 2 * ffn, generator=gen, device="cuda").to(dtype)
    for probs in (None, torch.rand(full.size(0), device="cuda")):
        expect, gp = K.gmm_swiglu_grad(full, w2, fc1, probs, whole, 1)
        mine = None if probs is None else probs[own].contiguous()
        d, gp_own = K.gmm_swiglu_grad(full[own].contiguous(), w2, fc1[own].contiguous(), mine, counts, 1)
        assert torch.equal(d, expect[own])
        assert probs is None or torch.equal(gp_own, gp[own])
