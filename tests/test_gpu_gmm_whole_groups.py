"""Launches split on rows that deal whole groups out to single XCDs (at least 16 groups of at most 8 row tiles, from six rounds of
tiles on): every kernel that can run such a launch, on whole numbers, so the sums are exact.  The workspace is the caller's, so
the test can read from the tile table in it that this is what the launch did."""
import ctypes

import pytest
import torch

from mindspeed_amd import _lib
from mindspeed_amd.ops._kernels import K

pytestmark = pytest.mark.gpu

# 32 groups of three row tiles, the third a 64-row one, a 128-row one or a full one, and rows past the last offset: with 17
# column panels 1632 tiles, six rounds being 1536
COUNTS = [(513, 576, 577, 640, 641, 700, 767, 768)[(5 * g) % 8] for g in range(32)]
REST, RED, COLS = 70, 72, 17 * 256
ROWS = sum(COUNTS)


def _operands(dtype):
    gen = torch.Generator(device="cuda").manual_seed(4)
    ints = lambda *s: torch.randint(-1, 2, s, generator=gen, device="cuda").to(dtype)
    return ints(ROWS + REST, RED), ints(len(COUNTS), RED, COLS), torch.tensor(COUNTS, device="cuda")


def _exact(x, w):
    parts = [a.float() @ b.float() for a, b in zip(x[:ROWS].split(COUNTS), w)]
    return torch.cat(parts + [torch.zeros(REST, w.size(2), device="cuda")])


def _call(name, workspace_size, *args):
    """The entry point with a workspace of its own, whose table must hold lists (its fourth word: where they lie)."""
    lib = _lib.load()
    need = ctypes.c_size_t(0)
    _lib.check(workspace_size(lib, ctypes.byref(need)), "workspace size")
    work = torch.zeros(need.value, dtype=torch.uint8, device="cuda")
    _lib.check(getattr(lib, name)(_lib.stream_ptr(work.device), *args, work.data_ptr(), work.numel()), name)
    torch.cuda.synchronize()
    assert int(work[:16].view(torch.int32)[3]) > 0, "no lists in the table"


def _rows_size(lib, out):
    return lib.ms_gmm_workspace_size(len(COUNTS), ROWS + REST, 0, out)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("transposed", [False, True])
def test_grouped_matmul(transposed, dtype):
    x, w, gl = _operands(dtype)
    if transposed:
        w = w.transpose(1, 2).contiguous().transpose(1, 2)
    want, code = _exact(x, w), _lib.dtype_code(dtype, "x")
    for out_dtype, out_code in ((dtype, code), (torch.float32, _lib.MS_FP32)):
        y = torch.full((ROWS + REST, COLS), float("nan"), dtype=out_dtype, device="cuda")
        for accumulate in (0, 1) if out_dtype == torch.float32 else (0,):
            _call("ms_gmm", _rows_size, x.data_ptr(), *x.stride(), w.data_ptr(), *w.stride(), y.data_ptr(), COLS, gl.data_ptr(), 1, 0,
                  len(COUNTS), ROWS + REST, RED, COLS, code, out_code, accumulate)
            assert torch.equal(y.float(), want * (1 + accumulate))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activation_in_the_epilogue(dtype):
    x, w, gl = _operands(dtype)
    w = w * 0.0625                              # gate values of the size an activation meets, still exact
    probs = torch.rand(ROWS + REST, device="cuda")
    ffn, code = COLS // 2, _lib.dtype_code(dtype, "x")
    fc1, act = (torch.full((ROWS + REST, n), float("nan"), dtype=dtype, device="cuda") for n in (COLS, ffn))
    _call("ms_gmm_swiglu", _rows_size, x.data_ptr(), *x.stride(), w.data_ptr(), *w.stride(), fc1.data_ptr(), COLS, act.data_ptr(), ffn,
          probs.data_ptr(), _lib.MS_FP32, gl.data_ptr(), 1, len(COUNTS), ROWS + REST, RED, ffn, code)
    assert torch.equal(fc1.float(), _exact(x, w)) and torch.equal(act, K.swiglu(fc1, probs))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activation_backward_in_the_epilogue(dtype):
    dy, w, gl = _operands(dtype)
    w2 = w.transpose(1, 2).contiguous()         # [E, ffn, hidden]
    wt = w2.transpose(1, 2)
    gen = torch.Generator(device="cuda").manual_seed(5)
    fc1 = torch.randn(ROWS + REST, 2 * COLS, generator=gen, device="cuda").to(dtype)
    probs = torch.rand(ROWS + REST, device="cuda")
    d_fc1, gp = torch.full_like(fc1, float("nan")), torch.full_like(probs, float("nan"))
    _call("ms_gmm_swiglu_grad", lambda lib, out: lib.ms_gmm_swiglu_grad_workspace_size(len(COUNTS), ROWS + REST, COLS, out),
          dy.data_ptr(), *dy.stride(), w2.data_ptr(), *wt.stride(), fc1.data_ptr(), 2 * COLS, probs.data_ptr(), _lib.MS_FP32,
          d_fc1.data_ptr(), 2 * COLS, gp.data_ptr(), gl.data_ptr(), 1, len(COUNTS), ROWS + REST, RED, COLS, _lib.dtype_code(dtype, "dy"))
    want, want_p = K.swiglu_grad(_exact(dy, wt).to(dtype), fc1, probs)
    assert torch.equal(d_fc1, want)
    # 4352 products of the same fp32 terms in two orders: 2^-24 of the sum of magnitudes per addition, in a tree of 64 columns a
    # leaf and 68 leaves over 64 lanes at most 64 + 8 additions deep on either side
    gate, up = fc1.float().chunk(2, dim=1)
    mag = (_exact(dy, wt) * torch.nn.functional.silu(gate) * up).abs().sum(dim=1)
    assert bool(((gp - want_p).abs() <= 2 * 72 * 2 ** -24 * mag).all())
