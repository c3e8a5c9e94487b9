"""The native side of the ops (csrc_host/launch.cpp) against the Python functions of the same names: equal results, equal
errors, and the same calls left to the dispatcher."""
import threading
from types import SimpleNamespace

import pytest
import torch

from mindspeed_amd import _lib, flop_counter
from mindspeed_amd.ops import _kernels as kernels
from mindspeed_amd.ops._kernels import K

pytestmark = pytest.mark.gpu


def _inputs():
    gen = torch.Generator(device="cuda").manual_seed(1)
    r = lambda *s, dtype=torch.bfloat16: torch.randn(*s, generator=gen, device="cuda").to(dtype)
    u = lambda *s: torch.rand(*s, generator=gen, device="cuda")
    i = SimpleNamespace(counts=torch.tensor([30, 0, 64, 6], device="cuda"), x=r(100, 64), w=r(4, 64, 128), dy=r(100, 128),
                        tokens=r(50, 72), index=torch.randint(0, 4, (50, 2), generator=gen, device="cuda"), probs=u(50, 2),
                        rmap=u(50, 6) < 0.4, mprobs=u(50, 6), p100=u(100), out=torch.zeros(4, 64, 128, device="cuda"),
                        acc=torch.ones(4, 64, 128, device="cuda"))
    i.permuted, i.rid, _, _ = kernels._permute(i.tokens, i.index, 100, 4, False, False)
    i.rows = int(i.rmap.sum()) + 3
    i.mperm, i.mrid, i.mflat, _, _ = kernels._routing_map_permute_probs(i.tokens, i.rmap, None, i.rows, False)
    i.gp = u(i.rows)
    return i


# (op, its arguments out of _inputs()): nothing runs on the device while the tests are collected
CALLS = {
    "gmm": lambda i: ("gmm", i.x, i.w, i.counts, 0, 1),
    "gmm_fp32_offsets": lambda i: ("gmm", i.x.float(), i.w.float(), i.counts.cumsum(0), 0, 0),
    "gmm_reduction": lambda i: ("gmm", i.x.t(), i.dy, i.counts, 2, 1),
    "gmm_transposed": lambda i: ("gmm", i.dy, i.w.transpose(1, 2), i.counts, 0, 1),
    "gmm_out": lambda i: ("gmm_out", i.x.t(), i.dy, i.counts, 2, 1, i.out, False),
    "gmm_out_accumulate": lambda i: ("gmm_out", i.x.t(), i.dy, i.counts, 2, 1, i.acc, True),
    "gmm_backward": lambda i: ("gmm_backward", i.dy, i.x, i.w, i.counts, 1, torch.empty_like(i.w), False),
    "gmm_backward_accumulate": lambda i: ("gmm_backward", i.dy, i.x, i.w, i.counts.cumsum(0), 0, i.acc, True),
    "gmm_swiglu": lambda i: ("gmm_swiglu", i.x, i.w, i.counts, 1, None, True),
    "gmm_swiglu_probs_no_fc1": lambda i: ("gmm_swiglu", i.x, i.w, i.counts, 1, i.p100, False),
    "permute": lambda i: ("moe_token_permute", i.tokens, i.index, 100, 4, True, True),
    "permute_int32": lambda i: ("moe_token_permute", i.tokens, i.index.int(), 90, 0, False, True),
    "permute_top1": lambda i: ("moe_token_permute", i.tokens, i.index[:, 0].contiguous(), 50, 4, False, False),
    "permute_grad": lambda i: ("moe_token_permute_grad", i.permuted, i.rid, 50, 2),
    "unpermute": lambda i: ("moe_token_unpermute", i.permuted, i.rid, None, 50, 2),
    "unpermute_probs": lambda i: ("moe_token_unpermute", i.permuted, i.rid, i.probs.half(), 50, 2),
    "unpermute_grad": lambda i: ("moe_token_unpermute_grad", i.permuted, i.tokens, i.rid, i.probs, 50, 2, 100),
    "unpermute_grad_half_probs": lambda i: ("moe_token_unpermute_grad", i.permuted, i.tokens, i.rid, i.probs.half(), 50, 2, 100),
    "unpermute_grad_marked": lambda i: ("moe_token_unpermute_grad", i.mperm, i.tokens, i.mrid, i.mprobs, 50, 6, i.rows, i.mflat),
    "unpermute_grad_more_rows": lambda i: ("moe_token_unpermute_grad", i.permuted, i.tokens, i.rid, None, 50, 2, 130),
    "swiglu": lambda i: ("swiglu", i.dy, None),
    "swiglu_probs": lambda i: ("swiglu", i.dy, i.p100),
    "swiglu_grad": lambda i: ("swiglu_grad", i.x, i.dy, None),
    "swiglu_grad_probs": lambda i: ("swiglu_grad", i.x, i.dy, i.p100.half()),
    "routing_map_permute": lambda i: ("routing_map_permute_probs", i.tokens, i.rmap, i.mprobs, i.rows, False),
    "routing_map_permute_no_probs": lambda i: ("routing_map_permute_probs", i.tokens, i.rmap, None, i.rows, False),
    "routing_map_probs_grad": lambda i: ("routing_map_probs_grad", i.mrid, i.gp, 50, 6),
}


def _flat(result):
    return [result] if isinstance(result, torch.Tensor) else list(result)


@pytest.mark.parametrize("case", CALLS)
def test_equals_the_python_function(case):
    name, *args = CALLS[case](_inputs())
    native = (kernels._native if kernels._native is not None else kernels._load_native())[name]
    clones = [a.clone(memory_format=torch.preserve_format) if isinstance(a, torch.Tensor) else a for a in args]
    want, got = kernels._DEVICE_FNS[name](*clones), native(*args)
    if name == "gmm_out":
        assert got is True and want is None
        want, got = clones[5], args[5]
    if name == "gmm_backward":
        want, got = (want, clones[5]), (got, args[5])
    for a, b in zip(_flat(want), _flat(got)):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)
    assert len(_flat(want)) == len(_flat(got))


def test_errors_are_those_of_the_python_function():
    x, gl = torch.randn(8, 16, device="cuda"), torch.tensor([4, 4], device="cuda")
    with pytest.raises(TypeError, match="should be bfloat16, float16 or float32"):
        K.gmm(x.double(), torch.randn(2, 16, 8, device="cuda").double(), gl, 0, 1)
    with pytest.raises(TypeError, match="should be bfloat16, float16 or float32"):
        K.swiglu(x.double(), None)
    with pytest.raises(_lib.MindSpeedAmdError, match=r"ms_gmm failed \(status -?\d+\): ms_gmm: group_type"):
        K.gmm(x, torch.randn(2, 16, 8, device="cuda"), gl, 1, 1)
    rid = torch.zeros(16, dtype=torch.int32, device="cuda")
    with pytest.raises(_lib.MindSpeedAmdError, match="ms_moe_token_permute_grad failed"):
        K.moe_token_permute_grad(x, rid, 8, 0)


def test_which_calls_are_plain():
    kernels._load_native()
    from mindspeed_amd import _host

    class Sub(torch.Tensor):
        pass
    t = torch.zeros(2, device="cuda")
    for args in ((t, 1, None, True), (torch.nn.Parameter(t), "a", 2.0), ([t, t], (t,)), (t, torch.zeros(2)),
                 (t.as_subclass(Sub),), ([t, torch.zeros(2)],), (torch.zeros(2, device="meta"),), ()):
        assert _host.plain(args) == kernels._plain_arguments(args)
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode() as mode:
        assert not _host.plain((t,))
        x = mode.from_tensor(torch.zeros(8, 16, device="cuda"))
        y = K.gmm(x, mode.from_tensor(torch.zeros(2, 16, 8, device="cuda")), mode.from_tensor(torch.tensor([4, 4], device="cuda")), 0, 1)
        assert y.shape == (8, 8)


def test_a_recorder_still_sees_the_calls():
    name, *args = CALLS["gmm"](_inputs())
    with flop_counter.record(timing=False) as rec:
        K.gmm(*args)
    assert [c[0] for c in rec.calls] == ["gmm_fwd"]


def test_current_stream_and_threads():
    """Every call goes to the caller's current stream, also from several threads at once."""
    name, *args = CALLS["gmm"](_inputs())
    want = K.gmm(*args)
    torch.cuda.synchronize()
    out = {}

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            x = args[0].clone()
            for _ in range(20):
                y = K.gmm(x, *args[1:])
            s.synchronize()
            out[i] = torch.equal(y, want)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert out == {i: True for i in range(4)}
