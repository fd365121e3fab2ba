"""Code that a user puts into the block -- a subclass's step, an instance's or a patched class's forward, a hook, a parametrization,
another callable as the operator -- runs: the fused paths of MHFFNLayer stand in for its own steps only."""
import pytest
import torch
from torch import nn
from torch.nn.utils import parametrize

from flashmhf_amd import FlashMLPMoE, MHFFNLayer
from flashmhf_amd.mhffn_layer import RMSNorm

H, dh, E, de = 2, 64, 3, 32


class Subclass(MHFFNLayer):
    def heads_and_gate(self, x):
        self.calls.append("heads_and_gate")
        return super().heads_and_gate(x)


class Double(nn.Module):
    def forward(self, w):
        return 2 * w


def _make(cls=MHFFNLayer):
    torch.manual_seed(0)
    layer = cls(H * dh, H, E, de, apply_rmsnorm=True)
    layer.calls = []
    return layer


def _wrapped(layer, name, f):
    return lambda *a: (layer.calls.append(name), f(*a))[1]


def _subclass(monkeypatch):
    return _make(Subclass)


def _instance_step(monkeypatch):
    layer = _make()
    layer.heads_and_gate = _wrapped(layer, "step", layer.heads_and_gate)
    return layer


def _patched_step(monkeypatch):
    layer, f = _make(), MHFFNLayer.heads_and_gate
    monkeypatch.setattr(MHFFNLayer, "heads_and_gate", lambda self, x: (layer.calls.append("step"), f(self, x))[1])
    return layer


def _instance_forward(child):
    def make(monkeypatch):
        layer = _make()
        m = getattr(layer, child)
        m.forward = _wrapped(layer, child, m.forward)
        return layer
    return make


def _patched_forward(cls):
    def make(monkeypatch):
        layer, f = _make(), cls.forward
        monkeypatch.setattr(cls, "forward", lambda self, *a: (layer.calls.append(cls), f(self, *a))[1])
        return layer
    return make


def _hook(child):
    def make(monkeypatch):
        layer = _make()
        getattr(layer, child).register_forward_hook(lambda *a: layer.calls.append(child))
        return layer
    return make


def _child_subclass(monkeypatch):
    class Linear(nn.Linear):
        def forward(self, x):
            layer.calls.append("linear")
            return super().forward(x)
    layer = _make()
    layer.w_self_2 = Linear(H * dh, H * dh, bias=False)
    return layer


def _function_op(monkeypatch):
    layer = _make()
    op = layer.op
    del layer.op
    layer.op = _wrapped(layer, "op", op)
    return layer


def _parametrized(monkeypatch):
    layer = _make()
    parametrize.register_parametrization(layer, "V", Double())
    layer.parametrizations.V[0].register_forward_hook(lambda *a: layer.calls.append("V"))
    return layer


CHILDREN = ("w_self", "w_self_2", "q_norm", "op")
CUSTOM = [_subclass, _instance_step, _patched_step, _child_subclass, _function_op, _parametrized,
          *(_instance_forward(c) for c in CHILDREN), *(_hook(c) for c in CHILDREN),
          *(_patched_forward(c) for c in (nn.Linear, RMSNorm, FlashMLPMoE))]


def test_a_plain_block_is_its_own():
    assert _make()._stock_steps()
    layer = MHFFNLayer(H * dh, H, E, de)
    assert layer._stock_steps()
    layer.q_norm = lambda q: q
    assert not layer._stock_steps()
    assert not MHFFNLayer(H * dh, H, E, de, bias=True)._stock_steps()


@pytest.mark.parametrize("make", CUSTOM)
def test_a_block_with_code_of_the_users_is_not(make, monkeypatch):
    assert not make(monkeypatch)._stock_steps()


@pytest.mark.gpu
@pytest.mark.parametrize("make", CUSTOM)
@pytest.mark.parametrize("grad", [False, True])
def test_code_of_the_users_runs_once(make, grad, monkeypatch):
    layer = make(monkeypatch).to("cuda:0").to(torch.bfloat16)
    x = torch.randn(2, 24, H * dh, generator=torch.Generator().manual_seed(1)).bfloat16().to("cuda:0").requires_grad_(grad)
    layer.calls.clear()
    y = layer(x)
    assert len(layer.calls) == (2 if nn.Linear in layer.calls else 1), layer.calls      # (two projections)
    assert y.isfinite().all() and (not grad or torch.autograd.grad(y.sum(), x)[0].isfinite().all())


@pytest.mark.gpu
def test_an_own_head_norm_takes_part():
    layer = _make().to("cuda:0").to(torch.bfloat16)
    x = torch.randn(2, 24, H * dh, device="cuda:0").bfloat16()
    layer.q_norm.forward = torch.zeros_like
    with torch.no_grad():
        assert not layer(x).any()       # O = sum_e R_e (silu(0) * 0) V


@pytest.mark.gpu
@pytest.mark.parametrize("norm", [lambda: RMSNorm((H, dh), 0.5), lambda: RMSNorm((dh,), 0.5), lambda: RMSNorm((dh,)), lambda: RMSNorm((1, dh), 0.5)])
@pytest.mark.parametrize("grad", [False, True])
def test_a_head_norm_in_place_of_the_block_s_is_the_one_that_runs(norm, grad):
    """Its epsilon (which outweighs the rows here) and its weight, in the block's node and in its steps, as in torch's operations."""
    dev, (B, S) = "cuda:0", (2, 24)
    layer = _make()
    layer.q_norm = norm()
    with torch.no_grad():
        layer.q_norm.weight.uniform_(0.5, 1.5, generator=torch.Generator().manual_seed(2))
    layer = layer.to(dev).to(torch.bfloat16)
    x = (torch.randn(B, S, H * dh, generator=torch.Generator().manual_seed(1)) * 0.25).bfloat16().to(dev).requires_grad_(grad)
    results = []
    for how in ("block", "steps", "torch"):
        if how == "steps":
            layer.w_self.register_forward_hook(lambda *a: None)
        layer.fused_prologue = how != "torch"
        y = layer(x)
        results.append([y, *torch.autograd.grad(y, [x, *layer.parameters()], torch.ones_like(y))] if grad else [y])
    for a, b, ref in zip(*results):
        for got in (a, b):
            # the two sides round bfloat16 intermediates at other places (2^-9 each, some ten of them)
            assert (got - ref).float().norm() <= 2e-2 * ref.float().norm()
