"""The block as one native node (flashmhf_amd/csrc/mhffn_torch.cpp) against the same block taken step by step, which a forward
hook on a projection brings back: the same kernels and library products, so every output and gradient is the same bit for
bit."""
import gc

import pytest
import torch

from flashmhf_amd.mhffn_layer import MHFFNLayer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,H,Hk,dh,E,de,rms", [(1, 1, 2, 2, 64, 1, 32, True), (2, 33, 4, 2, 96, 32, 32, False),
                                                  (3, 70, 4, 4, 128, 3, 96, True)])
@pytest.mark.parametrize("needs_dx", [True, False])
def test_one_node_block_is_the_stepwise_block(B, S, H, Hk, dh, E, de, rms, needs_dx):
    dev = "cuda:0"
    torch.manual_seed(S)
    layer = MHFFNLayer(H * dh, H, E, de, Hk, apply_rmsnorm=rms).to(dev).to(torch.bfloat16)
    x = torch.randn(B, S, H * dh, device=dev).bfloat16().requires_grad_(needs_dx)
    g = torch.randn(B, S, H * dh, device=dev).bfloat16()
    leaves = dict(layer.named_parameters())
    if needs_dx:
        leaves["x"] = x
    assert layer._one_node(x)
    results = []
    for stepwise in (False, True):
        if stepwise:
            layer.w_self.register_forward_hook(lambda *a: None)
            assert not layer._one_node(x)
        y = layer(x)
        grads = torch.autograd.grad(y, list(leaves.values()), g)
        with torch.no_grad():
            assert torch.equal(layer(x), y)
        results.append({"y": y, **dict(zip(leaves, grads))})
    for name, a in results[0].items():
        b = results[1][name]
        assert a.dtype == b.dtype and a.shape == b.shape, name
        assert torch.equal(a, b), name


def _products(f):
    """What f() returns and how many matrix products it ran."""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        out = f()
    return out, sum(e.count for e in prof.key_averages() if e.key == "aten::mm")


EXPERTS, PROLOGUE, PROJECTIONS = {"K", "U", "V"}, {"router", "q_norm.weight"}, {"w_self.weight", "w_self_2.weight"}


@pytest.mark.parametrize("rms", [True, False])
@pytest.mark.parametrize("needs_dx", [True, False])
@pytest.mark.parametrize("trained", [EXPERTS, PROLOGUE, PROJECTIONS, {"w_self.weight"}, {"w_self_2.weight"}, {"K"}, EXPERTS | PROLOGUE,
                                     EXPERTS | PROLOGUE | PROJECTIONS, set()])
@pytest.mark.parametrize("by", ["frozen", "named"])
def test_what_nobody_asks_for_is_not_computed(rms, needs_dx, trained, by):
    """Gradients of some of the block's tensors: the others frozen, or not named in torch.autograd.grad.  The same values as with
    the steps, no more matrix products, and no more memory kept between forward and backward."""
    dev, B, S, H, dh, E, de = "cuda:0", 2, 24, 2, 64, 3, 32
    torch.manual_seed(0)
    layer = MHFFNLayer(H * dh, H, E, de, apply_rmsnorm=rms).to(dev).to(torch.bfloat16)
    params = dict(layer.named_parameters())
    for name, p in params.items():
        p.requires_grad_(by == "named" or name in trained)
    x = torch.randn(B, S, H * dh, device=dev).bfloat16().requires_grad_(needs_dx or by == "named")
    dY = torch.randn_like(x)
    asked = [p for name, p in params.items() if name in trained] + [x] * needs_dx
    if not asked:
        pytest.skip("nothing to ask for")
    results = []
    for stepwise in (False, True):
        if stepwise:
            layer.w_self.register_forward_hook(lambda *a: None)
        layer(x)
        gc.collect()
        before = torch.cuda.memory_allocated()
        y = layer(x)
        kept = torch.cuda.memory_allocated() - before
        grads, products = _products(lambda: torch.autograd.grad(y, asked, dY))
        results.append((grads, products, kept, y))
    (ga, na, ka, ya), (gb, nb, kb, yb) = results
    assert torch.equal(ya, yb) and all(torch.equal(a, b) for a, b in zip(ga, gb))
    assert na == nb, (na, nb)
    assert ka <= kb, (ka, kb)
