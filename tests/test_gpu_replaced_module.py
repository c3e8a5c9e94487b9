"""Callers that put a module of their own behind ``GMMFunction.builder`` / ``builder2`` are asked for every product: by the gradient
accumulation fusion's backward pass and by the single-rank layer."""
import pytest
import torch

from mindspeed_amd.dispatcher import dispatch_mlp_combine
from mindspeed_amd.ops import gmm as gmm_ops
from mindspeed_amd.ops import npu_gmm, npu_gmm_v2

pytestmark = pytest.mark.gpu


class _Asked(gmm_ops._RawGmmModule):
    """The built-in products, counted; the input's gradient comes back doubled."""

    def __init__(self):
        self.calls = []

    def npu_gmm(self, *args):
        self.calls.append("npu_gmm")
        return gmm_ops._RawGmmModule.npu_gmm(*args)

    def npu_gmm_backward(self, *args):
        self.calls.append("npu_gmm_backward")
        (dx,), dw, dbias = gmm_ops._RawGmmModule.npu_gmm_backward(*args)
        return [2 * dx], dw, dbias

    def npu_gmm_backward_fusion(self, *args):
        self.calls.append("npu_gmm_backward_fusion")
        (dx,), dw, dbias = gmm_ops._RawGmmModule.npu_gmm_backward_fusion(*args)
        return [2 * dx], dw, dbias


class _OnlyFusion(gmm_ops._RawGmmModule):
    """One method replaced, the others inherited."""

    def __init__(self):
        self.calls = []

    npu_gmm_backward_fusion = _Asked.npu_gmm_backward_fusion


class _Loads:
    def __init__(self, module):
        self.module = module

    def load(self):
        return self.module


def _rand(*shape, seed=0, dtype=torch.bfloat16):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, generator=gen, device="cuda").to(dtype)


@pytest.mark.parametrize("cls", [_Asked, _OnlyFusion])
@pytest.mark.parametrize("name,op", [("builder", npu_gmm), ("builder2", npu_gmm_v2)])
def test_gradient_accumulation_fusion(name, op, cls, monkeypatch):
    x, gy = _rand(300, 64), _rand(300, 72, seed=1)
    counts = torch.tensor([100, 0, 200], device="cuda")
    groups = counts.cumsum(0) if op is npu_gmm else counts

    def step():
        w = _rand(3, 64, 72, seed=2).requires_grad_(True)
        w.main_grad = torch.ones(3, 64, 72, device="cuda")
        leaf = x.clone().requires_grad_(True)
        y = op(leaf, w, group_list=groups, gemm_fusion=True, original_weight=w)
        (dx,) = torch.autograd.grad(y, leaf, gy)
        return y.detach(), dx, w.main_grad

    y, dx, grad = step()
    module = cls()
    monkeypatch.setattr(gmm_ops.GMMFunction, name, _Loads(module))
    y2, dx2, grad2 = step()
    assert module.calls == (["npu_gmm"] if cls is _Asked else []) + ["npu_gmm_backward_fusion"]
    assert torch.equal(y, y2) and torch.equal(2 * dx, dx2) and torch.equal(grad, grad2)


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("how", ["builder", "method"])
def test_single_rank_layer(how, grad, monkeypatch):
    x, w1, w2 = _rand(40, 64), _rand(4, 64, 48, seed=1), _rand(4, 24, 64, seed=2)
    index = torch.arange(80, device="cuda").view(40, 2) % 4
    probs = torch.rand(40, 2, device="cuda").bfloat16()

    def layer():
        leaves = [t.clone().requires_grad_(grad) for t in (x, w1, w2)]
        with torch.set_grad_enabled(grad):
            y = dispatch_mlp_combine(leaves[0], index, probs, leaves[1:], fuse_activation=False)
        return [y.detach(), *(torch.autograd.grad(y, leaves[1:], torch.ones_like(y)) if grad else ())]

    expect = layer()
    module = _Asked()
    if how == "builder":
        monkeypatch.setattr(gmm_ops.GMMFunction, "builder2", _Loads(module))
    else:                                                # the built-in module's own method replaced
        monkeypatch.setattr(gmm_ops._RawGmmModule, "npu_gmm", staticmethod(_counted(module, gmm_ops._RawGmmModule.npu_gmm)))
    got = layer()
    assert module.calls.count("npu_gmm") == 2
    assert module.calls.count("npu_gmm_backward") == (2 if grad and how == "builder" else 0)
    assert torch.equal(expect[0], got[0])
    if grad:                                             # (the second matmul's doubled dX reaches the first one's weight)
        assert torch.equal(expect[2], got[2]) and torch.equal((2 if how == "builder" else 1) * expect[1], got[1])


def _counted(module, built_in):
    def npu_gmm(*args):
        module.calls.append("npu_gmm")
        return built_in(*args)
    return npu_gmm
