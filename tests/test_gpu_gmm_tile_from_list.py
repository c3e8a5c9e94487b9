"""Grouped matmuls of up to 64 groups, whose workgroups find their tiles in the group list by themselves, against the same
groups with empty ones added behind them up to 70, which go through the tile table.  A tile's sums do not depend on how it
was found, so the results are equal bit for bit; only the fp32 weight gradient may take tiles of another kind with more
groups, which add up in another order (at most 2e-6 of the sum of magnitudes for the fewer than 2200 products here)."""
import pytest
import torch

from mindspeed_amd.ops.gmm import gmm_raw

pytestmark = pytest.mark.gpu

PADDED = 70

# rows per group: remainders on both sides of the small tiles' edges, empty groups, one group, as many as a wavefront has
# lanes, many row tiles
COUNTS = {
    "edges": [1, 0, 63, 64, 65, 127, 128, 129, 255, 256, 257, 320],
    "one": [300],
    "empty_ends": [0, 0, 700, 0, 5, 0],
    "all_empty": [0, 0, 0],
    "lanes": [(37 * g) % 90 for g in range(64)],
    "long": [1400, 3, 2100],
}
SHAPES = {"fast": (torch.bfloat16, 192, 520), "fast_fp16": (torch.float16, 64, 256), "unaligned": (torch.bfloat16, 100, 259),
          "fp32": (torch.float32, 72, 200)}


def _lists(counts, rest, counted, device):
    """The group list, and the same with empty groups behind it; ``rest`` rows belong to no group."""
    gl = torch.tensor(counts, dtype=torch.int64)
    pad = torch.zeros(PADDED - len(counts), dtype=torch.int64)
    if not counted:
        gl = gl.cumsum(0)
        pad = pad + gl[-1]
    return gl.to(device), torch.cat([gl, pad]).to(device), int(sum(counts)) + rest


def _both(shape, gl, gl_pad, m, counted):
    dtype, k, n = SHAPES[shape]
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(m, k, generator=gen, device="cuda").to(dtype)
    w = torch.randn(gl.numel(), k, n, generator=gen, device="cuda").to(dtype)
    dy = torch.randn(m, n, generator=gen, device="cuda").to(dtype)
    w_pad = torch.cat([w, w.new_zeros(PADDED - gl.numel(), k, n)])
    kind = 1 if counted else 0
    assert torch.equal(gmm_raw(x, w, gl, 0, kind), gmm_raw(x, w_pad, gl_pad, 0, kind))
    assert torch.equal(gmm_raw(dy, w.transpose(1, 2), gl, 0, kind), gmm_raw(dy, w_pad.transpose(1, 2), gl_pad, 0, kind))
    dw, dw_pad = gmm_raw(x.t(), dy, gl, 2, kind), gmm_raw(x.t(), dy, gl_pad, 2, kind)[:gl.numel()]
    if dtype == torch.float32:
        assert bool(((dw - dw_pad).abs() <= 2e-6 * gmm_raw(x.abs().t(), dy.abs(), gl, 2, kind)).all())
    else:
        assert torch.equal(dw, dw_pad)


@pytest.mark.parametrize("counted", [True, False], ids=["counts", "offsets"])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("counts", COUNTS)
def test_same_tiles_as_from_the_table(counts, shape, counted):
    for rest in (0, 190):
        gl, gl_pad, m = _lists(COUNTS[counts], rest, counted, "cuda")
        if m:
            _both(shape, gl, gl_pad, m, counted)


def test_group_lists_that_run_backwards_or_past_the_rows():
    """Negative counts read as zero, offsets never run backwards, and neither leads past the rows."""
    for values, counted in (([5, -3, 200, 1 << 40, 7], True), ([100, 40, -8, 250, 1 << 40, 260], False)):
        gl = torch.tensor(values, dtype=torch.int64, device="cuda")
        pad = torch.zeros(PADDED - len(values), dtype=torch.int64, device="cuda")
        _both("fast", gl, torch.cat([gl, pad]), 333, counted)
        _both("fp32", gl, torch.cat([gl, pad]), 333, counted)
