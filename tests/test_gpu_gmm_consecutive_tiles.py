"""Launches split on rows whose XCDs take consecutive tiles of the whole launch: shares equal in number or in cost, rows past the
last offset behind them, shares that the launch has too few workgroups for, divided last rounds, tails in parts.  Whole numbers, so
the sums are exact; the output starts as NaN, so a tile that nobody takes shows.  The workspace is the caller's and the rule can be
evaluated on the host, so every case checks that it takes the way that it is there for."""
import ctypes

import pytest
import torch

from mindspeed_amd import _lib

CUS = 256
RED = 72              # one whole and one partial K step
# way the tiles are found, column tiles, reduction, rows per group, rows behind the groups
CASES = {
    # found in the group list
    "odd_numbers": ("list, by number", 3, RED, [700, 5, 0, 256, 1281], 0),
    "divided_last_round": ("list, by number", 15, RED, [1280, 1024, 1150, 768, 256, 1000], 90),
    "few_small_tiles_between": ("list, by number", 29, RED, [2048 + 30 * g for g in range(8)], 300),       # 8 rounds, 4 of 71 small
    "a_fifth_small_tiles_between": ("list, eighths", 52, RED, [1024 + 3 * g + 1 for g in range(8)], 0),
    "many_small_tiles_between": ("list, eighths", 90, RED, [257, 300, 520, 256, 70, 513, 1] * 2, 0),
    "seven_row_tiles_short_reduction": ("list, by number", 12, 3072, [1700 + g for g in range(8)], 10),
    "six_row_tiles_long_reduction": ("list, eighths", 12, 3080, [1500 + g for g in range(8)], 10),
    "nine_row_tiles_short_reduction": ("list, by number", 12, 2384, [2100, 1800, 2300, 2200], 0),
    "nine_row_tiles_long_reduction": ("list, eighths", 12, 2392, [2100, 1800, 2300, 2200], 0),
    "sixteen_groups_one_large": ("list, by number", 12, RED, [2600] + [250] * 15, 0),
    "fifteen_groups_one_large": ("list, eighths", 12, RED, [2600] + [250] * 14, 0),
    # from the table
    "seventy_groups": ("table, by number", 8, RED, [300 + g for g in range(70)], 33),
    "seventy_groups_of_one_round": ("table, eighths", 4, RED, [200, 100] * 35, 0),
    "sixteen_groups_of_112_tiles": ("table, by cost", 8, 136, [3584 + 256 * (g % 3 - 1) for g in range(16)], 0),
    "sixteen_groups_of_more": ("table, eighths", 8, 136, [3584 + 256 * (g % 3 - 1) for g in range(15)] + [3600], 0),
    "sixteen_large_groups": ("table, eighths", 13, 72, [2560] * 16, 0),
    "tails_in_parts": ("table, by number in parts", 16, 4168, [1024 + 10 * (g % 2) for g in range(8)], 5),
    "shares_by_cost": ("table, by cost", 28, RED, [2305] + [230 + 57 * g for g in range(19)], 130),          # seven rounds
    "shares_by_cost_one_block": ("table, by cost", 110, RED, [1024 + 7 * g for g in range(8)], 0),        # 17 rounds
    "shares_by_cost_long_reduction": ("table, by cost", 80, 4168, [1024 + 7 * g for g in range(8)], 0),
    "too_few_workgroups": ("table, too few workgroups", 28, RED, [1] * 30 + [256 * 90], 40),              # a share of small tiles only is too long
    "only_small_tiles": ("table, by cost", 20, RED, [64, 1, 128, 100] * 75, 0),                           # more groups than get lists of their own
    "whole_groups": ("per-XCD lists", 20, RED, [700] * 32, 0),
    "empty": ("table, eighths", 60, RED, [0] * 70, 1000),
}


def takes_together(name, from_list):
    _, col_tiles, red, counts, _ = CASES[name]
    out = ctypes.c_int(-1)
    _lib.check(_lib.load().msi_gmm_takes_together((ctypes.c_int64 * len(counts))(*counts), len(counts), red, col_tiles * 256 - 8,
                                                  from_list, CUS, ctypes.byref(out)), "msi_gmm_takes_together")
    return bool(out.value)


@pytest.mark.parametrize("name", CASES)
def test_the_rule_takes_the_case_as_named(name):
    way = CASES[name][0]
    if way != "per-XCD lists":
        assert takes_together(name, way.startswith("list")) == (not way.endswith("eighths"))


def test_bad_arguments_are_refused():
    out, rows = ctypes.c_int(0), (ctypes.c_int64 * 1)(-1)
    lib = _lib.load()
    for args in ((None, 1, 8, 8, 1, CUS), (rows, 1, 8, 8, 1, CUS), (rows, 0, 8, 8, 1, CUS), (rows, 1, 8, 0, 1, CUS)):
        assert lib.msi_gmm_takes_together(*args, ctypes.byref(out)) != 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", CASES)
def test_every_tile_once(name, dtype):
    assert torch.cuda.get_device_properties(0).multi_processor_count == CUS
    way, col_tiles, red, counts, rest = CASES[name]
    cols, rows, G = col_tiles * 256 - 8, sum(counts), len(counts)
    gen = torch.Generator(device="cuda").manual_seed(6)
    ints = lambda *s: torch.randint(-1, 2, s, generator=gen, device="cuda").to(dtype)
    x, w, gl = ints(rows + rest, red), ints(G, red, cols), torch.tensor(counts, device="cuda")
    want = torch.cat([a.float() @ b.float() for a, b in zip(x[:rows].split(counts), w)] + [torch.zeros(rest, cols, device="cuda")])
    want = want.to(dtype)                       # (whole numbers below 2^24 in fp32, rounded once, as the kernel's sums are)
    lib, code, need = _lib.load(), _lib.dtype_code(dtype, "x"), ctypes.c_size_t(0)
    sizes = (G, rows + rest, red, cols, 0, code, code, 0)
    _lib.check(lib.ms_gmm_workspace_size_split(*sizes, ctypes.byref(need)), "workspace size")
    for weight in (w, w.transpose(1, 2).contiguous().transpose(1, 2)):
        y = torch.full((rows + rest, cols), float("nan"), dtype=dtype, device="cuda")
        work = torch.zeros(need.value, dtype=torch.uint8, device="cuda")
        _lib.check(lib.ms_gmm(_lib.stream_ptr(work.device), x.data_ptr(), *x.stride(), weight.data_ptr(), *weight.stride(), y.data_ptr(),
                              y.stride(0), gl.data_ptr(), 1, 0, G, rows + rest, red, cols, code, code, 0, work.data_ptr(), work.numel()),
                   "ms_gmm")
        assert torch.equal(y, want)
        # the table's first words: slots (0: there is no table), entries, split tails, lists, .., tiles in order, shares by cost
        slots, _, tails, lists, _, _, _, _, in_order, by_cost = work[:40].view(torch.int32).tolist()
        if slots == 0:
            took = "list, by number" if takes_together(name, True) else "list, eighths"
        elif lists:
            took = "per-XCD lists"
        elif in_order:
            took = "table, by cost" if by_cost else "table, by number in parts" if tails else "table, by number"
        else:
            took = "table, too few workgroups" if takes_together(name, False) else "table, eighths"
        assert took == way
