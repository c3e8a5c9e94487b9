"""The fp32 grouped matmul in 32 x 32 tiles with the reduction split over four wavefronts, at the edges of its tiles, blocks and
quarters, against the products in 64 bits.  Sums of at most 300 fp32 products of N(0, 1) values in four chains are off by
some 1e-7 of their size; 2e-6 of the largest possible magnitude sum |a||b| leaves the rounding of every partial sum in."""
import pytest
import torch

from mindspeed_amd.ops.gmm import gmm_raw

pytestmark = pytest.mark.gpu

COUNTS = {"edges": [1, 31, 0, 32, 33, 65], "short": [3, 1, 2, 0, 1, 1], "mixed": [7, 8, 9, 130, 40, 257]}


def _close(got, want, bound):
    assert bool(((got.double() - want).abs() <= 2e-6 * bound + 1e-30).all())


def _rows(x, w, counts):
    out, mag, at = [], [], 0
    for g, c in enumerate(counts):
        out.append(x[at:at + c].double() @ w[g].double())
        mag.append(x[at:at + c].double().abs() @ w[g].double().abs())
        at += c
    tail = torch.zeros(x.size(0) - at, w.size(2), dtype=torch.float64, device=x.device)
    return torch.cat(out + [tail]), torch.cat(mag + [tail])


@pytest.mark.parametrize("k", [4, 8, 12, 28, 36, 100, 256, 300, 30])      # (30: not in quads, the general kernel)
@pytest.mark.parametrize("n", [1, 31, 33, 72])
@pytest.mark.parametrize("counts", COUNTS)
def test_split_on_rows(counts, k, n):
    counts = COUNTS[counts]
    gen = torch.Generator(device="cuda").manual_seed(k * 100 + n)
    m = sum(counts) + 5
    wide = torch.randn(m, k + 12, generator=gen, device="cuda")
    gl = torch.tensor(counts, device="cuda")
    w = torch.randn(len(counts), k, n, generator=gen, device="cuda")
    wt = w.transpose(1, 2).contiguous().transpose(1, 2)
    for x in (wide[:, :k].contiguous(), wide[:, :k], wide[:, 1:k + 1]):      # plain, strided rows, off the 16-byte grid
        want, mag = _rows(x, w, counts)
        for weight in (w, wt):
            y = torch.full((m, n), float("nan"), device="cuda")
            gmm_raw(x, weight, gl, 0, 1, out=y)
            _close(y, want, mag)
            gmm_raw(x, weight, gl, 0, 1, out=y, accumulate=True)
            _close(y, 2 * want, 2 * mag)


@pytest.mark.parametrize("k,n", [(1, 1), (31, 33), (64, 100), (130, 32)])
@pytest.mark.parametrize("counts", COUNTS)
def test_split_on_the_reduction(counts, k, n):
    counts = COUNTS[counts]
    gen = torch.Generator(device="cuda").manual_seed(k * 100 + n)
    m = sum(counts) + 3
    x = torch.randn(m, k, generator=gen, device="cuda")
    dy = torch.randn(m, n, generator=gen, device="cuda")
    gl = torch.tensor(counts, device="cuda")
    xs, ys = x[:sum(counts)].split(counts), dy[:sum(counts)].split(counts)
    want = torch.stack([a.double().t() @ b.double() for a, b in zip(xs, ys)])
    mag = torch.stack([a.double().abs().t() @ b.double().abs() for a, b in zip(xs, ys)])
    y = torch.full((len(counts), k, n), float("nan"), device="cuda")
    gmm_raw(x.t(), dy, gl, 2, 1, out=y)
    _close(y, want, mag)
    gmm_raw(x.t(), dy, gl, 2, 1, out=y, accumulate=True)
    _close(y, 2 * want, 2 * mag)
