"""Operands laid out backwards (a negative stride in one matrix dim), which a caller of the C ABI may pass: torch tensors have
none.  Kernels that address a tile by unsigned 32-bit offsets from its first element cannot take them.  Whole numbers, so every
sum is exact."""
import ctypes

import pytest
import torch

from mindspeed_amd import _lib

pytestmark = pytest.mark.gpu

COUNTS = [33, 0, 64, 7]
M, REST, KDIM, N = sum(COUNTS), 3, 64, 72


def _matrix(t, backwards):
    """(address of element (0, 0), strides) of the matrices t [..., r, c], dim `backwards` of the two (None: neither) read from
    its end."""
    strides, first = [t.stride(-2), t.stride(-1)], 0
    if backwards is not None:
        first = (t.size(backwards - 2) - 1) * strides[backwards]
        strides[backwards] = -strides[backwards]
    return t.data_ptr() + first * t.element_size(), strides


def _gmm(x, x_back, w, w_back, out, group_type):
    lib = _lib.load()
    gl = torch.tensor(COUNTS, device="cuda")
    (m, k), n = (x.shape if group_type == 0 else x.shape[::-1]), w.size(-1)
    xp, xs = _matrix(x, x_back)
    wp, ws = _matrix(w, w_back)
    code = _lib.dtype_code(x.dtype, "x")
    need = ctypes.c_size_t(0)
    _lib.check(lib.ms_gmm_workspace_size(len(COUNTS), m, group_type, ctypes.byref(need)), "ms_gmm_workspace_size")
    work = _lib.workspace(need.value, x.device)
    _lib.check(lib.ms_gmm(_lib.stream_ptr(x.device), xp, *xs, wp, w.stride(0) if group_type == 0 else 0, *ws, out.data_ptr(), n,
                          gl.data_ptr(), 1, group_type, len(COUNTS), m, k, n, code, code, 0, work.data_ptr(), work.numel()), "ms_gmm")
    torch.cuda.synchronize()
    return out


def _numbers(gen, dtype, *shape):
    return torch.randint(-3, 4, shape, generator=gen, device="cuda").to(dtype)


def _seen(t, backwards):
    return t.double() if backwards is None else t.double().flip(backwards - 2)


# which dims run backwards: (of x, of w as it is stored, w stored transposed)
FORMS = {"rows of x": (0, None, False), "reduction of w": (None, 0, False), "columns of w": (None, 1, True), "both": (0, 0, False),
         "both, w transposed": (0, 1, True)}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", FORMS)
def test_split_on_rows(form, dtype):
    x_back, w_back, transposed = FORMS[form]
    gen = torch.Generator(device="cuda").manual_seed(len(form))
    x = _numbers(gen, dtype, M + REST, KDIM)
    w = _numbers(gen, dtype, len(COUNTS), KDIM, N)
    if transposed:
        w = w.transpose(1, 2).contiguous().transpose(1, 2)
    out = _gmm(x, x_back, w, w_back, torch.full((M + REST, N), float("nan"), dtype=dtype, device="cuda"), 0)
    parts = _seen(x, x_back)[:M].split(COUNTS)
    want = torch.cat([a @ b for a, b in zip(parts, _seen(w, w_back))] + [torch.zeros(REST, N, dtype=torch.float64, device="cuda")])
    assert torch.equal(out, want.to(dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("x_back,w_back", [(1, None), (None, 0), (1, 0)])
def test_split_on_the_reduction(x_back, w_back, dtype):
    gen = torch.Generator(device="cuda").manual_seed(7)
    x = _numbers(gen, dtype, M, KDIM).t()
    dy = _numbers(gen, dtype, M, N)
    out = _gmm(x, x_back, dy, w_back, torch.full((len(COUNTS), KDIM, N), float("nan"), dtype=dtype, device="cuda"), 2)
    xs, ys = _seen(x, x_back).t().split(COUNTS), _seen(dy, w_back).split(COUNTS)
    want = torch.stack([a.t() @ b for a, b in zip(xs, ys)])
    assert torch.equal(out, want.to(dtype))


def test_the_fused_forms_refuse_them():
    """The kernels with the activation in their epilogue come in the vector-access form only."""
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(9)
    x, w = _numbers(gen, torch.bfloat16, M, KDIM), _numbers(gen, torch.bfloat16, len(COUNTS), KDIM, 2 * N)
    act, gl = torch.empty(M, N, dtype=x.dtype, device="cuda"), torch.tensor(COUNTS, device="cuda")
    xp, xs = _matrix(x, 0)
    need = ctypes.c_size_t(0)
    _lib.check(lib.ms_gmm_workspace_size(len(COUNTS), M, 0, ctypes.byref(need)), "ms_gmm_workspace_size")
    work = _lib.workspace(need.value, x.device)
    rc = lib.ms_gmm_swiglu(_lib.stream_ptr(x.device), xp, *xs, w.data_ptr(), *w.stride(), None, 2 * N, act.data_ptr(), N, None, 0,
                           gl.data_ptr(), 1, len(COUNTS), M, KDIM, N, _lib.MS_BF16, work.data_ptr(), work.numel())
    assert rc != 0 and b"vector-access layout" in lib.ms_last_error()
