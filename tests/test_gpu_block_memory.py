"""Memory of the block's backward: a gradient of the tokens is given back as soon as the step that reads it has run."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rms", [True, False])
def test_backward_keeps_three_gradients_of_the_tokens(rms):
    """At the end there are the prologue's incoming and outgoing gradient and that of x; never the operator's incoming one as well."""
    from flashmhf_amd import MHFFNLayer
    T, hid = 16384, 1024      # (one token slice and one part: no partial sums)
    m = MHFFNLayer(hid, 8, 11, 352, 8, apply_rmsnorm=rms).to(DEV, torch.bfloat16)
    x = torch.randn(4, T // 4, hid, device=DEV).bfloat16().requires_grad_()
    dy = torch.randn_like(x)
    for _ in range(2):
        y = m(x)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        grads = torch.autograd.grad(y, [x, *m.parameters()], dy)
        torch.cuda.synchronize()
        peak = torch.cuda.max_memory_allocated() - before
        one = T * hid * 2
        weights = sum(g.numel() * g.element_size() for g in grads[1:])
        gates = 4 * T * 8 * 11                         # dR
        del y, grads
    print("peak", peak, "gradients", (peak - weights - gates) / one, flush=True)
    assert peak <= 3.5 * one + weights + gates
