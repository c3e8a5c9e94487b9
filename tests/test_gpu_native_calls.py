"""The native side of the ops (csrc_host/launch.cpp) against the Python functions of the same names: equal results, equal
errors, and the same calls left to the dispatcher."""
import threading

import pytest
import torch

from mindspeed_amd import _lib, flop_counter
from mindspeed_amd.ops import _kernels as kernels
from mindspeed_amd.ops._kernels import K

pytestmark = pytest.mark.gpu


def _calls():
    gen = torch.Generator(device="cuda").manual_seed(1)
    r = lambda *s, dtype=torch.bfloat16: torch.randn(*s, generator=gen, device="cuda").to(dtype)
    counts = torch.tensor([30, 0, 64, 6], device="cuda")
    x, w, dy = r(100, 64), r(4, 64, 128), r(100, 128)
    tokens, index = r(50, 72), torch.randint(0, 4, (50, 2), generator=gen, device="cuda")
    permuted, rid, _, _ = kernels._permute(tokens, index, 100, 4, False, False)
    probs = torch.rand(50, 2, generator=gen, device="cuda")
    rmap = torch.rand(50, 6, generator=gen, device="cuda") < 0.4
    rows = int(rmap.sum()) + 3
    mperm, mrid, mflat, _, _ = kernels._routing_map_permute_probs(tokens, rmap, None, rows, False)
    mprobs = torch.rand(50, 6, generator=gen, device="cuda")
    out, acc = torch.zeros(4, 64, 128, device="cuda"), torch.ones(4, 64, 128, device="cuda")
    return [("gmm", x, w, counts, 0, 1), ("gmm", x.float(), w.float(), counts.cumsum(0), 0, 0), ("gmm", x.t(), dy, counts, 2, 1),
            ("gmm", dy, w.transpose(1, 2), counts, 0, 1),
            ("gmm_out", x.t(), dy, counts, 2, 1, out, False), ("gmm_out", x.t(), dy, counts, 2, 1, acc, True),
            ("gmm_swiglu", x, w, counts, 1, None, True), ("gmm_swiglu", x, w, counts, 1, torch.rand(100, device="cuda"), False),
            ("moe_token_permute", tokens, index, 100, 4, True, True), ("moe_token_permute", tokens, index.int(), 90, 0, False, True),
            ("moe_token_permute", tokens, index[:, 0].contiguous(), 50, 4, False, False),
            ("moe_token_permute_grad", permuted, rid, 50, 2),
            ("moe_token_unpermute", permuted, rid, None, 50, 2), ("moe_token_unpermute", permuted, rid, probs.half(), 50, 2),
            ("moe_token_unpermute_grad", permuted, tokens, rid, probs, 50, 2, 100),
            ("moe_token_unpermute_grad", permuted, tokens, rid, probs.half(), 50, 2, 100),
            ("moe_token_unpermute_grad", mperm, tokens, mrid, mprobs, 50, 6, rows, mflat),
            ("moe_token_unpermute_grad", permuted, tokens, rid, None, 50, 2, 130),
            ("swiglu", dy, None), ("swiglu", dy, torch.rand(100, device="cuda")), ("swiglu_grad", x, dy, None),
            ("swiglu_grad", x, dy, torch.rand(100, device="cuda").half()),
            ("routing_map_permute_probs", tokens, rmap, mprobs, rows, False), ("routing_map_permute_probs", tokens, rmap, None, rows, False),
            ("routing_map_probs_grad", mrid, torch.rand(rows, device="cuda"), 50, 6)]


def _flat(result):
    return [result] if isinstance(result, torch.Tensor) else list(result)


@pytest.mark.parametrize("i", range(len(_calls()) if torch.cuda.is_available() else 25))
def test_equals_the_python_function(i):
    name, *args = _calls()[i]
    native = (kernels._native if kernels._native is not None else kernels._load_native())[name]
    clones = [a.clone(memory_format=torch.preserve_format) if isinstance(a, torch.Tensor) else a for a in args]
    want, got = kernels._DEVICE_FNS[name](*clones), native(*args)
    if name == "gmm_out":
        assert got is True and want is None
        want, got = clones[5], args[5]
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
    name, *args = _calls()[0]
    with flop_counter.record(timing=False) as rec:
        K.gmm(*args)
    assert [c[0] for c in rec.calls] == ["gmm_fwd"]


def test_current_stream_and_threads():
    """Every call goes to the caller's current stream, also from several threads at once."""
    name, *args = _calls()[0]
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
