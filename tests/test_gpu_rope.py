"""The decoder's rotary positions in one pass each way against the element-wise operations they stand for (bfloat16, every
product and sum rounded): the same values, forward and backward, also for gradients of other strides."""
import pytest
import torch

from flashmhf_amd.mhffn_layer import _apply_rotary, _rotary

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,H,d", [(1, 1, 1, 16), (2, 37, 3, 96), (3, 130, 4, 64), (1, 257, 16, 128)])
@pytest.mark.parametrize("strided", [False, True])
def test_rope_is_the_element_wise_form(B, S, H, d, strided):
    from flashmhf_amd import _capi
    dev = "cuda:0"
    torch.manual_seed(S)
    qkv = torch.randn(B, S, 3 * H * d, device=dev).bfloat16()
    cos, sin = _rotary(S, d, 10000.0, torch.device(dev), torch.bfloat16)
    grads = [torch.randn(B, S, H, d + 2 * strided, device=dev).bfloat16()[..., :d].transpose(1, 2) for _ in range(3)]
    a, b = qkv.clone().requires_grad_(True), qkv.clone().requires_grad_(True)
    out = _capi.native().rope(a, cos, sin, H)
    q, k, v = b.view(B, S, 3, H, d).permute(2, 0, 3, 1, 4)
    ref = (_apply_rotary(q, cos, sin), _apply_rotary(k, cos, sin), v)
    for x, y in zip(out, ref):
        assert torch.equal(x, y) and x.stride() == y.stride()
    ga, gb = torch.autograd.grad(out, a, grads)[0], torch.autograd.grad(ref, b, grads)[0]
    assert torch.equal(ga, gb)
    with torch.no_grad():
        assert all(torch.equal(x, y) for x, y in zip(_capi.native().rope(a, cos, sin, H), out))
    only_v = torch.autograd.grad(_capi.native().rope(a, cos, sin, H)[2], a, grads[2])[0].view(B, S, 3, H, d)
    assert torch.equal(only_v[:, :, 2], grads[2].transpose(1, 2)) and not only_v[:, :, :2].any()
