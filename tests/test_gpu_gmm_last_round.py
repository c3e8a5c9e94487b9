"""Launches of few rounds of tiles divide the full tiles of their last, partly filled round into tiles of 128 or 64 rows.
The same groups inside a launch of many rounds run as whole tiles; a row's sums are formed in the same order either way,
so the results are equal bit for bit."""
import pytest
import torch

from mindspeed_amd.ops._kernels import K
from mindspeed_amd.ops.gmm import gmm_raw

pytestmark = pytest.mark.gpu

ROUND = 256           # compute units
K_DIM = 72            # one whole and one partial K step
# (column tiles, rows per group): tiles left for the last round 1, 5, 63, 64, 65, 127, 128 and 129 (whole again), behind no
# or one complete round, tails beside them, last tiles whose later parts hold no row, an empty group
CASES = {
    "one_tile": (1, [256]),
    "five": (5, [130]),
    "quarters_63": (9, [512, 0, 700, 192, 256]),
    "quarters_64_of_256_more": (16, [256 * 4] * 5),
    "quarters_beside_tails": (8, [256 * 3 + 60, 256 * 2 + 100, 190]),
    "halves_65": (13, [256 * 4, 129]),
    "halves_127_more": (1, [256 * 100 + 200, 256 * 282]),
    "halves_128": (8, [256 * 15, 250]),
    "whole_129": (3, [256 * 43]),
    "table_70_groups": (4, [0] * 60 + [256, 300, 40, 0, 511, 255, 129, 128, 64, 1]),
    "rows_behind_the_groups": (6, [300, 500]),
}


def _problem(cols, counts, rest):
    """Operands of the launch, and of one of at least seven rounds that begins with the same groups."""
    gen = torch.Generator(device="cuda").manual_seed(11)
    n, rows = cols * 256, sum(counts)
    more = (7 * ROUND // cols + 1) * 256
    x = torch.randn(rows + rest + more, K_DIM, generator=gen, device="cuda").bfloat16()
    w = torch.randn(len(counts) + 1, K_DIM, n, generator=gen, device="cuda").bfloat16()
    short = torch.tensor(counts, dtype=torch.int64, device="cuda")
    long = torch.tensor(counts + [rest + more], dtype=torch.int64, device="cuda")
    return x, w, short, long, rows


@pytest.mark.parametrize("name", CASES)
def test_equals_the_whole_tiles_of_a_long_launch(name):
    cols, counts = CASES[name]
    rest = 77 if name == "rows_behind_the_groups" else 0
    x, w, short, long, rows = _problem(cols, counts, rest)
    few = x[:rows + rest]
    wt = w.transpose(1, 2).contiguous().transpose(1, 2)
    for weight in (w, wt):
        y = torch.full((rows + rest, w.size(2)), float("nan"), dtype=x.dtype, device="cuda")
        gmm_raw(few, weight[:-1], short, 0, 1, out=y)
        whole = gmm_raw(x, weight, long, 0, 1)
        assert torch.equal(y[:rows], whole[:rows])
        assert bool((y[rows:] == 0).all())
    y32 = torch.full((rows + rest, w.size(2)), float("nan"), device="cuda")
    gmm_raw(few, w[:-1], short, 0, 1, out=y32)
    whole32 = torch.empty(x.size(0), w.size(2), device="cuda")
    gmm_raw(x, w, long, 0, 1, out=whole32)
    assert torch.equal(y32[:rows], whole32[:rows])


@pytest.mark.parametrize("name", ["five", "quarters_63", "halves_65", "halves_128"])
def test_fused_activation_forms(name):
    cols, counts = CASES[name]
    x, w, short, long, rows = _problem(2 * cols, counts, 0)      # (a fused tile holds 128 gate and 128 up columns)
    few = x[:rows]
    probs = torch.rand(x.size(0), device="cuda")
    fc1, act = K.gmm_swiglu(few, w[:-1], short, 1, probs[:rows], True)
    fc1_long, act_long = K.gmm_swiglu(x, w, long, 1, probs, True)
    assert torch.equal(fc1, fc1_long[:rows]) and torch.equal(act, act_long[:rows])
    w2 = w[:, :, :cols * 256].transpose(1, 2).contiguous()       # [E, ffn, hidden]
    fc1, fc1_long = fc1[:, :2 * cols * 256].contiguous(), fc1_long[:, :2 * cols * 256].contiguous()
    d, gp = K.gmm_swiglu_grad(few, w2[:-1], fc1, probs[:rows], short, 1)
    d_long, gp_long = K.gmm_swiglu_grad(x, w2, fc1_long, probs, long, 1)
    assert torch.equal(d, d_long[:rows]) and torch.equal(gp, gp_long[:rows])
