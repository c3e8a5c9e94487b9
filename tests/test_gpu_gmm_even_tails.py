"""A group whose last row tile would be a small one has its last two tiles share their rows: in long launches and in the one launch
of both gradients any, elsewhere one of two row tiles.  The same rows in groups that fill their tiles give the same bits, and every row is written once: the
outputs start as NaN, and rows behind the groups are zero."""
import pytest
import torch

from conftest import rel_l2
from mindspeed_amd.ops._kernels import K
from mindspeed_amd.ops.gmm import gmm_backward_raw, gmm_raw

pytestmark = pytest.mark.gpu

EDGES = [257, 288, 320, 321, 352, 384, 385, 511, 512, 513, 576, 577, 640, 641, 767, 768, 897]
# groups; by 12 column tiles: tiles from the group list, from a table, from per-XCD lists (equal groups)
GROUPS = {
    "list": EDGES + [1, 64, 65, 128, 0, 129, 256] + [25600],
    "table_of_many_rounds": EDGES + [40, 0, 100, 40960 + 17],
    "table_of_many_groups": [0, 300] * 20 + EDGES * 3 + [25600 + 60],
    "whole_groups_per_xcd": [300] * 128,
    "whole_groups_per_xcd_65_to_128": [560 + g % 80 for g in range(64)],
    "rows_behind_the_groups": EDGES + [25600 + 100],
}


def _rows(counts, k, rest=0):
    """The groups' rows, packed with `rest` more behind them and each filled up to whole tiles, and which of the latter they are."""
    whole = [(c + 255) // 256 * 256 for c in counts]
    gen = torch.Generator(device="cuda").manual_seed(len(counts) + k)
    full = torch.randn(sum(whole), k, generator=gen, device="cuda").bfloat16()
    begin = 0
    own = []
    for c, f in zip(counts, whole):
        own.append(torch.arange(begin, begin + c, device="cuda"))
        begin += f
    own = torch.cat(own)
    packed = torch.cat([full[own], torch.randn(rest, k, generator=gen, device="cuda").bfloat16()])
    return full, own, packed, torch.tensor(counts, device="cuda"), torch.tensor(whole, device="cuda")


@pytest.mark.parametrize("k", [72, 192])
@pytest.mark.parametrize("name", GROUPS)
def test_equals_tiles_that_are_full(name, k):
    n, counts = 12 * 256 - 16, GROUPS[name]
    rest = 333 if name == "rows_behind_the_groups" else 0
    full, own, x, short, whole = _rows(counts, k, rest)
    gen = torch.Generator(device="cuda").manual_seed(n)
    w = torch.randn(len(counts), k, n, generator=gen, device="cuda").bfloat16()
    for weight in (w, w.transpose(1, 2).contiguous().transpose(1, 2)):
        y = torch.full((x.size(0), n), float("nan"), dtype=x.dtype, device="cuda")
        gmm_raw(x, weight, short, 0, 1, out=y)
        assert torch.equal(y[:own.numel()], gmm_raw(full, weight, whole, 0, 1)[own])
        assert bool((y[own.numel():] == 0).all())
    ends = short.cumsum(0)
    y32 = torch.full((x.size(0), n), float("nan"), device="cuda")
    gmm_raw(x, w, ends, 0, 0, out=y32)
    whole32 = torch.empty(full.size(0), n, device="cuda")
    gmm_raw(full, w, whole, 0, 1, out=whole32)
    assert torch.equal(y32[:own.numel()], whole32[own])
    fc1, act = K.gmm_swiglu(x, w, short, 1, None, True)
    assert torch.equal(fc1, y) and torch.equal(act, K.swiglu(y, None))


# short launches: last rounds divided into parts of such tiles or not, small tiles of other groups beside them, whole or (from a
# reduction of 4096 on) with their reduction split
@pytest.mark.parametrize("cols,k,counts", [
    (1, 72, [300]), (3, 72, [257, 288, 320, 321, 384, 385, 5, 0, 640]), (12, 136, [300, 380] * 6), (16, 72, [1024, 330, 260] * 4),
    (7, 200, [290] * 70), (5, 4224, [300, 600, 350, 20]), (16, 8256, [512, 380, 600, 257])])
def test_groups_of_two_row_tiles_in_short_launches(cols, k, counts):
    n = cols * 256 - 40
    full, own, x, short, whole = _rows(counts, k)
    gen = torch.Generator(device="cuda").manual_seed(n)
    w = torch.randn(len(counts), k, n, generator=gen, device="cuda").bfloat16()
    two = torch.cat([torch.full((c,), 256 < c <= 384, device="cuda") for c in counts])
    for weight in (w, w.transpose(1, 2).contiguous().transpose(1, 2)):
        y = torch.full((x.size(0) + 2, n), float("nan"), dtype=x.dtype, device="cuda")
        gmm_raw(x, weight, short, 0, 1, out=y[:-2])
        expect = gmm_raw(full, weight, whole, 0, 1)[own]
        assert torch.equal(y[:-2][two], expect[two])
        if k < 4096:
            assert torch.equal(y[:-2], expect)
        assert rel_l2(y[:-2], expect) <= 4e-3               # (the sums of a split reduction are added in another order)
        assert bool(y[-2:].isnan().all())


@pytest.mark.parametrize("counts", [EDGES, [30, 0, 600, 1100], [300] * 20, EDGES * 4, [1024 + 13 * (g - 4) for g in range(8)]],
                         ids=["edges", "few", "20_equal", "68_groups", "8_ragged"])
def test_gradient_of_the_rows_in_one_launch_with_the_weight(counts):
    k, n = 5 * 256 + 64, 136
    full, own, grad, short, whole = _rows(counts, n)
    gen = torch.Generator(device="cuda").manual_seed(k)
    w = torch.randn(len(counts), k, n, generator=gen, device="cuda").bfloat16()
    x = torch.randn(own.numel(), k, generator=gen, device="cuda").bfloat16()
    dw, apart = torch.full_like(w, float("nan")), torch.empty_like(w)
    dx = gmm_backward_raw(grad, x, w, short, 1, dw)
    assert torch.equal(dx, gmm_raw(full, w.transpose(1, 2), whole, 0, 1)[own])
    gmm_raw(x.t(), grad, short, 2, 1, out=apart)
    assert torch.equal(dw, apart)
