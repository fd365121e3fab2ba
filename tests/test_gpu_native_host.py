"""The block as one native node (flashmhf_amd/csrc/mhffn_torch.cpp) against the same block taken step by step, which a forward
hook on a projection brings back: the same kernels and library products, so every output and gradient is the same bit for
bit."""
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
