"""dX and dW of one grouped matmul from one call: both products' tiles in one launch (from the group list, from two tables, with
per-XCD lists), either order, and what is left to two launches.  Whole numbers, so the sums are exact and one rounding away from
the reference; both outputs start as NaN (with accumulate: dW as whole numbers), so a tile that nobody takes shows."""
import ctypes

import pytest
import torch

from mindspeed_amd import _lib
from mindspeed_amd.ops import gmm as gmm_ops
from mindspeed_amd.ops._kernels import K

BF, HALF, FP32 = torch.bfloat16, torch.float16, torch.float32
# rows per group, rows behind the groups, k, n, dtype
CASES = {
    "one_row": ([1], 0, 8, 8, BF),
    "tile_edges": ([255, 256, 257, 0, 64, 65, 128, 129, 1], 3, 264, 520, BF),
    "one_tile_each": ([256] * 4, 0, 256, 256, HALF),
    "dw_first": ([3000, 1500], 0, 264, 72, BF),                    # more rows per group than dX has to reduce over
    "dw_first_empty_groups": ([0, 4000, 0, 0], 70, 136, 256, HALF),
    "sixteen_groups": ([130 + 9 * g for g in range(16)], 0, 520, 264, BF),
    "forty_eight_groups_many_rounds": ([300] * 48, 5, 1280, 1032, BF),
    "forty_nine_groups_few_rounds": ([100 + g for g in range(49)], 0, 520, 264, BF),
    "sixty_four_groups_tables": ([257 + (g % 5) for g in range(64)], 9, 3600, 136, BF),
    "sixty_four_equal_groups_lists": ([700] * 64, 0, 2056, 520, HALF),
    "sixty_five_groups": ([40 * (g % 3) for g in range(65)], 11, 264, 264, BF),
    "two_hundred_and_fifty_seven_groups": ([g % 70 for g in range(257)], 0, 136, 72, BF),
    "no_rows": ([0, 0, 0], 0, 64, 64, BF),
    "fp32": ([31, 32, 33, 0, 64, 1], 2, 36, 132, FP32),
    "fp32_dw_first": ([700, 600], 0, 64, 36, FP32),
    "fp32_quarters": ([128] * 8, 0, 256, 512, FP32),
    # two launches
    "odd_width": ([100, 57], 0, 70, 72, BF),
    "fp32_odd_width": ([100, 57], 0, 70, 72, FP32),
    "fp32_large": ([2000] * 2, 0, 2048, 2048, FP32),
}


def operands(name, seed=0):
    counts, behind, k, n, dtype = CASES[name]
    gen = torch.Generator().manual_seed(seed)
    m = sum(counts) + behind
    small = lambda *s: torch.randint(-2, 3, s, generator=gen).to(dtype).cuda()          # noqa: E731
    return small(m, n), small(m, k), small(len(counts), k, n), torch.tensor(counts, device="cuda")


def reference(grad, x, weight, counts):
    """Exact (whole numbers below 2^24), in fp32."""
    dx = torch.zeros(x.shape, dtype=FP32, device="cuda")
    dw = torch.zeros(weight.shape, dtype=FP32, device="cuda")
    begin = 0
    for g, rows in enumerate(counts.tolist()):
        part = slice(begin, begin + rows)
        dx[part] = grad[part].float() @ weight[g].float().t().contiguous()
        dw[g] = x[part].float().t().contiguous() @ grad[part].float()
        begin += rows
    return dx, dw


def call(grad, x, weight, group_list, list_type, dx, dw, accumulate):
    lib, (m, k), n, groups = _lib.load(), x.shape, weight.size(2), group_list.numel()
    dtype, dw_dtype = _lib.dtype_code(x.dtype, "x"), _lib.dtype_code(dw.dtype, "dw")
    need = ctypes.c_size_t(0)
    _lib.check(lib.msi_gmm_backward_workspace_size(groups, m, k, n, dtype, dw_dtype, accumulate, ctypes.byref(need)), "size")
    ws = torch.empty(need.value, dtype=torch.uint8, device="cuda")
    _lib.check(lib.msi_gmm_backward(
        _lib.stream_ptr(x.device), _lib.ptr(grad), *grad.stride(), _lib.ptr(x), *x.stride(), _lib.ptr(weight), *weight.stride(),
        _lib.ptr(dx), _lib.ptr(dw), _lib.ptr(group_list), list_type, groups, m, k, n, dtype, dw_dtype, accumulate, _lib.ptr(ws),
        ws.numel()), "msi_gmm_backward")


@pytest.mark.gpu
@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("accumulate", [False, True])
def test_both_gradients(name, accumulate):
    grad, x, weight, counts = operands(name)
    group_list = counts.cumsum(0) if accumulate else counts
    want_dx, want_dw = reference(grad, x, weight, counts)
    dx = torch.full_like(x, float("nan"))
    if accumulate:
        old = torch.arange(want_dw.numel(), device="cuda").remainder(7).view(want_dw.shape).float()
        dw, want_dw = old.clone(), want_dw + old
    else:
        dw = torch.full_like(weight, float("nan"))
    call(grad, x, weight, group_list, 0 if accumulate else 1, dx, dw, int(accumulate))
    assert torch.equal(dx, want_dx.to(dx.dtype))
    assert torch.equal(dw, want_dw.to(dw.dtype))


# operands that one of the two products, or neither, takes as they are
STRIDES = {
    "as_stored": lambda grad, x, weight: (grad, x, weight),
    "weight_along_k": lambda grad, x, weight: (grad, x, weight.transpose(1, 2).contiguous().transpose(1, 2)),
    "rows_of_wider": lambda grad, x, weight: (torch.cat([grad, grad], 1)[:, :grad.size(1)], torch.cat([x, x], 1)[:, x.size(1):], weight),
    "x_along_rows": lambda grad, x, weight: (grad, x.t().contiguous().t(), weight),
    "grad_expanded": lambda grad, x, weight: (grad[:1].expand(grad.size(0), -1), x, weight),
    "grad_every_other": lambda grad, x, weight: (torch.stack([grad, grad], 2)[:, :, 0], x, weight),
    "weight_one_element_on": lambda grad, x, weight: (grad, x, torch.cat([weight.new_zeros(1), weight.reshape(-1)])[1:].view(weight.shape)),
}


@pytest.mark.gpu
@pytest.mark.parametrize("form", STRIDES)
@pytest.mark.parametrize("name", ["tile_edges", "fp32"])
def test_operands_by_strides(name, form):
    grad, x, weight, counts = operands(name, seed=1)
    grad, x, weight = STRIDES[form](grad, x, weight)
    want_dx, want_dw = reference(grad, x, weight, counts)
    dw = torch.full(weight.shape, float("nan"), dtype=weight.dtype, device="cuda")
    dx = gmm_ops.gmm_backward_raw(grad, x, weight, counts, 1, dw)
    assert torch.equal(dx, want_dx.to(dx.dtype)) and torch.equal(dw, want_dw.to(dw.dtype))


@pytest.mark.gpu
def test_mistakes_keep_their_errors():
    grad, x, weight, counts = operands("tile_edges")
    dw = torch.empty_like(weight)
    with pytest.raises(TypeError, match="same dtype"):
        gmm_ops.gmm_backward_raw(grad.half(), x, weight, counts, 1, dw)
    with pytest.raises(ValueError, match="does not match"):
        gmm_ops.gmm_backward_raw(grad[1:], x, weight, counts, 1, dw)
    with pytest.raises(ValueError, match="contiguous tensor of the result's size"):
        gmm_ops.gmm_backward_raw(grad, x, weight, counts, 1, dw[:, 1:])
    with pytest.raises(ValueError, match="accumulate needs an fp32 out"):
        gmm_ops.gmm_backward_raw(grad, x, weight, counts, 1, dw, accumulate=True)
    with pytest.raises(TypeError, match="one-dimensional int64"):
        gmm_ops.gmm_backward_raw(grad, x, weight, counts.int(), 1, dw)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["tile_edges", "sixty_four_groups_tables", "fp32"])
def test_recorded_into_a_graph(name):
    grad, x, weight, counts = operands(name)
    dx, dw = torch.empty_like(x), torch.empty_like(weight)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        call(grad, x, weight, counts, 1, dx, dw, 0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        call(grad, x, weight, counts, 1, dx, dw, 0)
    for seed in range(3):                                 # new operands and group sizes at the same addresses
        again = operands(name, seed)
        for old, new in zip((grad, x, weight), again):
            old.copy_(new)
        counts.copy_(counts.flip(0))
        dx.fill_(float("nan"))
        dw.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        want_dx, want_dw = reference(grad, x, weight, counts)
        assert torch.equal(dx, want_dx.to(dx.dtype)) and torch.equal(dw, want_dw.to(dw.dtype))


def test_shapes_without_a_device():
    grad, x, weight = (torch.empty(s, dtype=BF, device="meta") for s in ((10, 24), (10, 16), (3, 16, 24)))
    group_list, dw = torch.empty(3, dtype=torch.int64, device="meta"), torch.empty(3, 16, 24, dtype=BF, device="meta")
    assert K.gmm_backward(grad, x, weight, group_list, 1, dw, False).shape == (10, 16)
    assert gmm_ops.gmm_backward_raw(grad, x, weight, group_list, 1, dw).shape == (10, 16)


@pytest.mark.parametrize("groups", [1, 16, 64, 256, 4096])
def test_the_workspace_holds_two_tables(groups):
    lib, need, plain = _lib.load(), ctypes.c_size_t(0), ctypes.c_size_t(0)
    _lib.check(lib.msi_gmm_backward_workspace_size(groups, 1000, 256, 512, _lib.MS_BF16, _lib.MS_BF16, 0, ctypes.byref(need)), "size")
    _lib.check(lib.ms_gmm_workspace_size(groups, 1000, 0, ctypes.byref(plain)), "size")
    assert need.value >= 2 * plain.value and plain.value % 256 == 0
    assert lib.msi_gmm_backward_workspace_size(groups, 1000, 256, 512, _lib.MS_BF16, _lib.MS_BF16, 0, None) != 0
