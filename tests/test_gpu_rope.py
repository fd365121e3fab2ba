"""The decoder's rotary positions in one pass each way against the element-wise operations they stand for (bfloat16, every
product and sum rounded): the same values, forward and backward, also for gradients of other strides."""
import pytest
import torch

from flashmhf_amd.mhffn_layer import CausalSelfAttention, _apply_rotary, _rotary
from tests.test_gpu_projection_callers import Memory, Wrapper

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


@pytest.mark.parametrize("B,S,H,d", [(1, 1, 1, 16), (2, 37, 3, 96)])
def test_derivatives_of_the_gradient_are_the_element_wise_forms(B, S, H, d):
    """create_graph: the gradient is a function of the outputs' gradients, and so on to any order (the map is linear)."""
    from flashmhf_amd import _capi
    dev = "cuda:0"
    torch.manual_seed(S)
    qkv = torch.randn(B, S, 3 * H * d, device=dev).bfloat16()
    cos, sin = _rotary(S, d, 10000.0, torch.device(dev), torch.bfloat16)
    grads = [torch.randn(B, H, S, d, device=dev).bfloat16() for _ in range(3)]
    v2, v3 = torch.randn_like(qkv), [torch.randn(B, H, S, d, device=dev).bfloat16() for _ in range(3)]
    results = []
    for native in (True, False):
        x, g = qkv.clone().requires_grad_(), [t.clone().requires_grad_() for t in grads]
        if native:
            out = _capi.native().rope(x, cos, sin, H)
        else:
            q, k, v = x.view(B, S, 3, H, d).permute(2, 0, 3, 1, 4)
            out = _apply_rotary(q, cos, sin), _apply_rotary(k, cos, sin), v
        dx, = torch.autograd.grad(out, x, g, create_graph=True)
        w = v2.clone().requires_grad_()
        dg = torch.autograd.grad(dx, g, w, create_graph=True)
        dw, = torch.autograd.grad(dg, w, v3)
        results.append([dx, *dg, dw])
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_gradient_penalty_through_attention(monkeypatch):
    """All terms of a second derivative, those behind q, k and v among them, against the element-wise rotary form (which tables
    of another shape bring back).  The attention itself is a stand-in of element-wise products: which of torch's attention
    kernels has a second derivative is not this module's business."""
    from flashmhf_amd import mhffn_layer
    from flashmhf_amd.mhffn_layer import CausalSelfAttention
    monkeypatch.setattr(mhffn_layer.F, "scaled_dot_product_attention", lambda q, k, v, is_causal: torch.tanh(q) * k * v)
    B, S, H, d = 2, 24, 2, 64
    torch.manual_seed(0)
    attn = CausalSelfAttention(H * d, H).to("cuda:0").to(torch.bfloat16)
    x = torch.randn(B, S, H * d, device="cuda:0").bfloat16().requires_grad_()
    cos, sin = _rotary(S, d, 10000.0, x.device, x.dtype)
    results = []
    for tables in ((cos, sin), (cos[None], sin[None])):
        dx, = torch.autograd.grad(attn(x, rope=tables).float().sum(), x, create_graph=True)
        results.append([dx, *torch.autograd.grad(dx.float().square().sum(), [x, *attn.parameters()])])
    for a, b in zip(*results):
        assert torch.equal(a, b)


def _both(x, tables, H, d):
    """The native call and the element-wise form."""
    from flashmhf_amd import _capi
    B, S, _ = x.shape
    q, k, v = x.view(B, S, 3, H, d).permute(2, 0, 3, 1, 4)
    return _capi.native().rope(x, *tables, H), (_apply_rotary(q, *tables), _apply_rotary(k, *tables), v)


@pytest.mark.parametrize("asked", [(0, 1, 2), (0,), (2,)])
def test_gradients_that_are_more_than_their_memory(asked):
    """Tangents (forward mode for the backward alone), batches, subclasses with code of their own: what the element-wise form gives."""
    from torch.autograd import forward_ad
    dev, (B, S, H, d) = "cuda:0", (2, 9, 3, 32)
    torch.manual_seed(0)
    tables = _rotary(S, d, 10000.0, torch.device(dev), torch.bfloat16)
    x = torch.randn(B, S, 3 * H * d, device=dev).bfloat16().requires_grad_()
    outs = [[o[i] for i in asked] for o in _both(x, tables, H, d)]
    dys, ts = ([torch.randn(B, H, S, d, device=dev).bfloat16() for _ in asked] for _ in range(2))
    with forward_ad.dual_level():
        got, want = (forward_ad.unpack_dual(torch.autograd.grad(o, x, [forward_ad.make_dual(*p) for p in zip(dys, ts)], retain_graph=True)[0])
                     for o in outs)
        assert torch.equal(got.primal, want.primal) and torch.equal(got.tangent, want.tangent)
    got, want = (torch.autograd.grad(o, x, [torch.stack(p) for p in zip(dys, ts)], is_grads_batched=True, retain_graph=True)[0] for o in outs)
    assert torch.equal(got, want)
    for cls in (Wrapper, Memory):
        got, want = (torch.autograd.grad(o, x, [cls.of(t) for t in dys], retain_graph=True)[0] for o in outs)
        assert isinstance(got, cls) and torch.equal(got.plain, want.plain)


@pytest.mark.parametrize("cls", [Wrapper, Memory])
def test_code_of_a_tensor_runs(cls):
    dev, (B, S, H, d) = "cuda:0", (2, 9, 3, 32)
    torch.manual_seed(0)
    tables = _rotary(S, d, 10000.0, torch.device(dev), torch.bfloat16)
    x = torch.randn(B, S, 3 * H * d, device=dev).bfloat16()
    _, want = _both(x, tables, H, d)
    got, _ = _both(cls.of(x), tables, H, d)
    assert all(isinstance(a, cls) and torch.equal(a.plain, b) for a, b in zip(got, want))


def test_a_subclass_is_carried_through():
    class Named(torch.Tensor):
        pass
    dev, (S, H, d) = "cuda:0", (9, 3, 32)
    attn = CausalSelfAttention(H * d, H).to(dev).to(torch.bfloat16)
    x = torch.randn(2, S, H * d, device=dev).bfloat16()
    y = attn(x.as_subclass(Named))
    assert type(y) is Named and torch.equal(y.as_subclass(torch.Tensor), attn(x))
