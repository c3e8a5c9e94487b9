"""Launches split on rows whose XCDs take consecutive tiles of the whole launch: shares equal in number or in cost, rows past the
last offset behind them, shares that the launch has too few workgroups for, divided last rounds.  Whole numbers, so the sums are
exact; the output starts as NaN, so a tile that nobody takes shows."""
import pytest
import torch

from mindspeed_amd.ops.gmm import gmm_raw

pytestmark = pytest.mark.gpu

RED = 72              # one whole and one partial K step
# (column tiles, rows per group, rows behind the groups)
CASES = {
    "odd_numbers": (3, [700, 5, 0, 256, 1281], 0),                                   # few rounds, found in the group list
    "divided_last_round": (15, [1280, 1024, 1150, 768, 256, 1000], 90),
    "few_small_tiles_between": (29, [2304 + 30 * g for g in range(8)], 300),         # 8 rounds, found in the group list
    "many_small_tiles_between": (90, [257, 300, 520, 256, 70, 513, 1] * 2, 0),      # as many as full ones: eighths
    "shares_by_cost": (40, [2305] + [30 + 37 * g for g in range(19)], 130),          # seven rounds, from the table
    "shares_by_cost_one_block": (110, [1024 + 7 * g for g in range(8)], 0),          # 14 rounds
    "too_few_workgroups": (30, [1] * 30 + [256 * 30], 40),                           # a share of small tiles only is too long
    "only_small_tiles": (20, [64, 1, 128, 100] * 75, 0),                             # more groups than get lists of their own
    "empty": (60, [0] * 70, 1000),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", CASES)
def test_every_tile_once(name, dtype):
    col_tiles, counts, rest = CASES[name]
    cols, rows = col_tiles * 256 - 8, sum(counts)
    gen = torch.Generator(device="cuda").manual_seed(6)
    ints = lambda *s: torch.randint(-1, 2, s, generator=gen, device="cuda").to(dtype)
    x, w, gl = ints(rows + rest, RED), ints(len(counts), RED, cols), torch.tensor(counts, device="cuda")
    want = torch.cat([a.float() @ b.float() for a, b in zip(x[:rows].split(counts), w)] + [torch.zeros(rest, cols, device="cuda")])
    for weight in (w, w.transpose(1, 2).contiguous().transpose(1, 2)):
        y = torch.full((rows + rest, cols), float("nan"), dtype=dtype, device="cuda")
        gmm_raw(x, weight, gl, 0, 1, out=y)
        assert torch.equal(y.float(), want)
