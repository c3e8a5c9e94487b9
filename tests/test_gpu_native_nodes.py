"""The native autograd nodes (csrc_host/launch.cpp: the index-form layer, the routing-map permute and unpermute) against the
Python functions that they stand for: equal results and gradients bit for bit, the same errors, and every call that something
else than autograd wants to see left to those functions."""
import threading

import pytest
import torch

from mindspeed_amd import _lib, dispatcher, flop_counter
from mindspeed_amd.dispatcher import dispatch_mlp_combine
from mindspeed_amd.ops import _kernels as kernels
from mindspeed_amd.ops import gmm as gmm_ops
from mindspeed_amd.ops import moe_permute_mask_map as mask_map

pytestmark = pytest.mark.gpu
BF, HALF, FP32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture
def taken(monkeypatch):
    """Names of the native forms that took a call, in order; ``taken.off()`` leaves every call to the Python functions."""
    class Taken(list):
        on = True

        def off(self):
            self.on = False
            return self

    names, real = Taken(), kernels.native_form

    def form(name, *args):
        out = real(name, *args) if names.on else None
        if out is not None:
            names.append(name)
        return out
    for module in (dispatcher, mask_map):
        monkeypatch.setattr(module, "native_form", form)
    return names


def layer_inputs(dtype=BF, pdtype=BF, tokens=37, hidden=72, experts=5, topk=2, ffn=40, index_dtype=torch.int64, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen, device="cuda")                                # noqa: E731
    index = torch.randint(0, experts, (tokens, topk), generator=gen, device="cuda").to(index_dtype)
    return [r(tokens, hidden).to(dtype), index, torch.rand(tokens, topk, generator=gen, device="cuda").to(pdtype),
            r(experts, hidden, 2 * ffn).to(dtype) * 0.1, r(experts, ffn, hidden).to(dtype) * 0.1]


def run_layer(args, wanted=(0, 2, 3, 4), grad=None, **kwargs):
    """(output, gradients of the wanted arguments) of one pass on fresh leaves of these values and strides."""
    leaves = [a.detach() for a in args]
    for i in wanted:
        leaves[i].requires_grad_(True)
    y = dispatch_mlp_combine(leaves[0], leaves[1], leaves[2], (leaves[3], leaves[4]), **kwargs)
    if not wanted:
        return [y]
    dy = torch.ones_like(y) if grad is None else grad(y)
    return [y.detach(), *torch.autograd.grad(y, [leaves[i] for i in wanted], dy)]


def equal(a, b):
    return len(a) == len(b) and all(x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y) for x, y in zip(a, b))


FORMS = {
    "bf16": {}, "fp16_fp32_probs": dict(dtype=HALF, pdtype=FP32), "fp32": dict(dtype=FP32, pdtype=FP32),
    "fp32_bf16_probs": dict(dtype=FP32, pdtype=BF), "int32": dict(index_dtype=torch.int32), "top1": dict(topk=1),
    "one_token": dict(tokens=1), "odd_sizes": dict(hidden=70, ffn=33), "fp32_odd_sizes": dict(dtype=FP32, pdtype=FP32, hidden=33, ffn=35),
}


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("wanted", [(0, 2, 3, 4), (3, 4), (0,), (2,), (3,), ()])
def test_layer_equals_the_ops(form, wanted, taken):
    args = layer_inputs(**FORMS[form])
    dy = lambda y: torch.randn(y.shape, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda").to(y.dtype)   # noqa: E731
    got = run_layer(args, wanted, dy)
    assert taken == ["layer"]
    taken.off()
    assert equal(got, run_layer(args, wanted, dy))


@pytest.mark.parametrize("form", FORMS)
def test_inference_equals_the_ops(form, taken):
    args = layer_inputs(**FORMS[form])
    with torch.no_grad():
        got = run_layer(args, ())
        assert taken == ["layer"]
        taken.off()
        assert equal(got, run_layer(args, ()))


STRIDES = {
    "tokens_of_wider": lambda a: [torch.cat([a[0], a[0]], 1)[:, :a[0].size(1)], *a[1:]],
    "tokens_expanded": lambda a: [a[0][:1].expand(a[0].shape), *a[1:]],
    "index_transposed": lambda a: [a[0], a[1].t().contiguous().t(), *a[2:]],
    "index_of_one_dim": lambda a: [a[0], a[1][:, 0], a[2][:, :1], *a[3:]],
    "probs_expanded": lambda a: [*a[:2], a[2][:1].expand(a[2].shape), *a[3:]],
    "weights_along_k": lambda a: [*a[:3], *(w.transpose(1, 2).contiguous().transpose(1, 2) for w in a[3:])],
    "every_other_expert": lambda a: [*a[:3], *(torch.stack([w, w], 1)[:, 0] for w in a[3:])],
    "every_other_element": lambda a: [*a[:3], *(torch.stack([w, w], -1)[..., 0] for w in a[3:])],
    "one_element_on": lambda a: [*a[:3], *(torch.cat([w.new_zeros(1), w.reshape(-1)])[1:].view(w.shape) for w in a[3:])],
}


@pytest.mark.parametrize("form", STRIDES)
@pytest.mark.parametrize("grads", [True, False])
def test_layer_by_strides(form, grads, taken):
    args = STRIDES[form](layer_inputs())
    passes = []
    for _ in range(2):
        with torch.set_grad_enabled(grads):
            passes.append(run_layer(args, (0, 2, 3, 4) if grads else (), lambda y: y.detach()[:1].expand(y.shape)))
        taken.off()
    assert equal(*passes)


def test_mistakes_keep_their_errors(taken):
    x, index, probs, w1, w2 = layer_inputs()
    for bad in ((x, index[1:], probs, w1, w2), (x, index.float(), probs, w1, w2), (x, index, probs, w1[1:], w2), (x, index, probs, w1, w2[:, 1:]),
                (x, index, probs.double(), w1, w2), (x.double(), index, probs, w1, w2), (x.half(), index, probs, w1, w2),
                (x, index, probs[1:], w1, w2), (x.cpu(), index, probs, w1, w2), (x, index, probs, w1[:, 1:], w2), (x[0], index, probs, w1, w2)):
        with pytest.raises(Exception) as first:
            dispatch_mlp_combine(*bad[:3], bad[3:], num_global_experts=5)
        taken.on = False
        with pytest.raises(first.type) as second:
            dispatch_mlp_combine(*bad[:3], bad[3:], num_global_experts=5)
        taken.on = True
        assert str(first.value) == str(second.value)
    assert taken == []


def mask_inputs(dtype=BF, pdtype=FP32, tokens=45, experts=6, hidden=40, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(tokens, hidden, generator=gen, device="cuda").to(dtype), torch.rand(tokens, experts, generator=gen, device="cuda") < 0.4,
            torch.rand(tokens, experts, generator=gen, device="cuda").to(pdtype))


def run_route(x, mask, probs, rows, drop=False, permute_probs=True, fused=False):
    x, mask, probs = x.detach().requires_grad_(True), mask.clone(), probs.detach().requires_grad_(True)
    permuted, permuted_probs, order = mask_map.permute(x, mask, probs=probs if permute_probs else None, num_out_tokens=rows, fused=fused,
                                                       drop_and_pad=drop)
    back = mask_map.unpermute(permuted, order, x.shape, probs=None if permute_probs else probs, routing_map=mask, drop_and_pad=drop)
    out = (back.float() ** 2).sum()
    if permute_probs:
        out = out + (permuted_probs.float() ** 2).sum()
    grads = torch.autograd.grad(out, (x, probs))
    return [permuted.detach(), order, back.detach(), *grads, *([permuted_probs.detach()] if permute_probs else [])]


@pytest.mark.parametrize("dtype,pdtype", [(BF, FP32), (BF, BF), (HALF, FP32), (FP32, FP32), (FP32, BF)])
@pytest.mark.parametrize("permute_probs", [True, False])
@pytest.mark.parametrize("drop,extra", [(False, 0), (False, 7), (True, 0)])
def test_routing_map_equals_the_functions(dtype, pdtype, permute_probs, drop, extra, taken):
    x, mask, probs = mask_inputs(dtype, pdtype)
    rows = 6 * 20 + 3 if drop else int(mask.sum()) + extra
    for fused in (False, True):
        taken.on = True
        got = run_route(x, mask, probs, rows, drop, permute_probs, fused)
        assert taken[-2:] == ["map_permute", "map_unpermute"]
        taken.off()
        want = run_route(x, mask, probs, rows, drop, permute_probs, fused)
        if extra:                                # (rows past the mask's entries come unwritten)
            got[0], want[0] = got[0][:-extra], want[0][:-extra]
            got[1], want[1] = got[1][:-extra], want[1][:-extra]
        assert equal(got, want)


def test_routing_map_calls_that_need_a_look(taken):
    x, mask, probs = mask_inputs()
    rows = int(mask.sum())
    assert mask_map.permute(x, mask)[0].shape == (rows, x.size(1))                # the count is read back
    with pytest.raises(RuntimeError, match="differs from routing_map shape"):
        mask_map.permute(x, mask, probs=probs[:, 1:], num_out_tokens=rows)
    with pytest.raises(RuntimeError, match="outside"):
        mask_map.permute(x, mask, num_out_tokens=mask.numel() + 1)
    assert taken == []
    permuted, _, order = mask_map.permute(x, mask, num_out_tokens=rows)
    assert taken == ["map_permute"]
    mask_map.unpermute(permuted, order.clone(), x.shape, routing_map=mask)        # an unknown index tensor is compared once
    mask_map.unpermute(permuted, order, x.shape, routing_map=mask.clone())
    assert taken == ["map_permute"]
    with pytest.raises(ValueError, match="not the token order"):
        mask_map.unpermute(permuted, order.flip(0), x.shape, routing_map=mask)
    order.flip(0).sort()
    mask[0] = ~mask[0]                                                            # the mask changed: its map is sorted afresh
    with pytest.raises((ValueError, AssertionError)):
        mask_map.unpermute(permuted, order, x.shape, routing_map=mask)


def test_saved_tensor_hooks_and_checkpoints(taken):
    args = layer_inputs()
    plain = run_layer(args)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.shape), t.cpu())[1], lambda t: t.cuda()):
        assert equal(run_layer(args), plain)
    assert len(seen) >= 10
    leaves = [a.detach().requires_grad_(a.is_floating_point()) for a in args]
    fn = lambda x, i, p, a, b: dispatch_mlp_combine(x, i, p, (a, b))             # noqa: E731
    y = torch.utils.checkpoint.checkpoint(fn, *leaves, use_reentrant=False)
    grads = torch.autograd.grad(y, [leaves[i] for i in (0, 2, 3, 4)], torch.ones_like(y))
    assert equal([y.detach(), *grads], plain) and set(taken) == {"layer"}
    x, mask, probs = mask_inputs()
    rows = int(mask.sum())
    plain = run_route(x, mask, probs, rows)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda()):
        assert equal(run_route(x, mask, probs, rows), plain)


def test_a_changed_saved_tensor_is_noticed(taken):
    args = layer_inputs()
    leaves = [a.detach().requires_grad_(a.is_floating_point()) for a in args]
    y = dispatch_mlp_combine(*leaves[:3], leaves[3:])
    with torch.no_grad():
        leaves[4].add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()
    y = dispatch_mlp_combine(*leaves[:3], leaves[3:])
    first = torch.autograd.grad(y, leaves[0], torch.ones_like(y), retain_graph=True)
    assert equal(first, torch.autograd.grad(y, leaves[0], torch.ones_like(y)))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y, leaves[0], torch.ones_like(y))


def test_transforms_and_subclasses_are_left_to_the_functions(taken):
    import torch.autograd.forward_ad as fwd

    x, index, probs, w1, w2 = layer_inputs()
    call = lambda t: dispatch_mlp_combine(t, index, probs, (w1, w2))             # noqa: E731
    with fwd.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        call(fwd.make_dual(x, torch.ones_like(x)))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: call(t).float().sum())(x)
    with pytest.raises(RuntimeError):
        torch.func.vmap(call)(torch.stack([x, x]))
    with torch.no_grad():
        dispatch_mlp_combine(x, index, probs, (w1, w2), fuse_activation=False)
    assert taken == ["layer"]

    class Sub(torch.Tensor):
        pass
    y = call(x.as_subclass(Sub))
    assert taken == ["layer"] and torch.equal(y.as_subclass(torch.Tensor), call(x))
    from torch._subclasses.fake_tensor import FakeTensorMode
    taken.clear()
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        assert call(mode.from_tensor(x)).shape == x.shape
    assert taken == []


def test_a_recorder_sees_every_op(taken, monkeypatch):
    args = layer_inputs()
    plain = run_layer(args)
    with flop_counter.record(timing=False) as rec:
        assert equal(run_layer(args), plain)
    names = [c[0] for c in rec.calls]
    assert sorted(names) == sorted(["permute", "gmm_fwd", "swiglu", "gmm_fwd", "unpermute", "unpermute_grad", "gmm_dw", "gmm_dx", "swiglu_grad",
                                    "gmm_dw", "gmm_dx", "permute_grad"])
    leaves = [a.detach().requires_grad_(a.is_floating_point()) for a in args]
    y = dispatch_mlp_combine(*leaves[:3], leaves[3:])
    with flop_counter.record(timing=False) as late:                              # between the two directions
        grads = torch.autograd.grad(y, [leaves[i] for i in (0, 2, 3, 4)], torch.ones_like(y))
    assert equal([y.detach(), *grads], plain)
    assert sorted(c[0] for c in late.calls) == sorted(["unpermute_grad", "gmm_dw", "gmm_dx", "swiglu_grad", "gmm_dw", "gmm_dx", "permute_grad"])
    for wanted in ((0,), (3,)):
        with flop_counter.record(timing=False):
            assert equal(run_layer(args, wanted), run_layer(args, wanted))
    monkeypatch.setattr(gmm_ops, "OVERLAP_WGRAD", True)
    taken.clear()
    assert equal(run_layer(args), plain) and taken == []


@pytest.mark.parametrize("wanted", [(3,), (3, 4), (0,), (2,), (0, 3)])
def test_a_recorder_around_the_backward_pass_alone(wanted, taken):
    """The native forward's nodes call the Python functions from the autograd thread, whichever gradients are wanted."""
    args = layer_inputs()
    plain = run_layer(args, wanted)
    leaves = [a.detach() for a in args]
    for i in wanted:
        leaves[i].requires_grad_(True)
    y = dispatch_mlp_combine(*leaves[:3], leaves[3:])
    with flop_counter.record(timing=False) as rec:
        grads = torch.autograd.grad(y, [leaves[i] for i in wanted], torch.ones_like(y))
    assert taken == ["layer", "layer"] and equal([y.detach(), *grads], plain)
    names = [c[0] for c in rec.calls]
    # (a matmul's gradients: by what lies in front of it and whether its weight is wanted)
    in_front = [0 in wanted, bool({0, 3} & set(wanted))]
    assert names.count("gmm_dx") == sum(in_front) and names.count("gmm_dw") == (3 in wanted) + (4 in wanted)


def test_a_failed_call_in_the_backward_pass(taken, monkeypatch):
    """The library's refusal reaches the caller as the package's error whichever thread met it."""
    args = layer_inputs()
    leaves = [a.detach().requires_grad_(a.is_floating_point()) for a in args]
    y = dispatch_mlp_combine(*leaves[:3], leaves[3:])

    def refuse(*_):
        raise _lib.MindSpeedAmdError("ms_swiglu_grad failed")
    monkeypatch.setitem(kernels._DEVICE_FNS, "swiglu_grad", refuse)
    with flop_counter.record(timing=False), pytest.raises(_lib.MindSpeedAmdError, match="ms_swiglu_grad failed"):
        y.sum().backward()


def test_threads_and_streams(taken):
    """Passes of several threads at once, each on a stream of its own, whose tensors are given back while the others run."""
    want = [run_layer(layer_inputs(seed=s)) for s in range(4)]
    torch.cuda.synchronize()
    failed = []

    def work(seed):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for _ in range(8):
                    got = run_layer(layer_inputs(seed=seed))
                    stream.synchronize()
                    if not equal(got, want[seed]):
                        failed.append(seed)
        except Exception as e:                                                   # noqa: BLE001
            failed.append(e)
    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
