"""What meets the projections' own products as it meets torch's linear layer: forward mode, batched gradients and tensors with code
of their own, in the forward call and in the backward alone."""
import warnings

import pytest
import torch
from torch.autograd import forward_ad

from flashmhf_amd import MHFFNDecoder, MHFFNLayer
from flashmhf_amd.mhffn_layer import OrderedProjection, Projection

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
B, S, H, dh, E, de = 2, 24, 2, 64, 3, 32


def _layer(**kw):
    torch.manual_seed(0)
    return MHFFNLayer(H * dh, H, E, de, apply_rmsnorm=True, **kw).to(DEV).to(torch.bfloat16)


def _lm_head():
    torch.manual_seed(0)
    return MHFFNDecoder(192, H * dh, 1, H, H, E, de).to(DEV).to(torch.bfloat16).lm_head


# (and torch's own layer, which says what is expected)
PROJECTIONS = {"torch": lambda: torch.nn.Linear(H * dh, 192, bias=False, device=DEV, dtype=torch.bfloat16), "w_self": lambda: _layer().w_self,
               "lm_head": _lm_head,
               "any order": lambda: Projection(H * dh, 192, bias=False, device=DEV, dtype=torch.bfloat16),
               "in order": lambda: OrderedProjection(H * dh, 192, bias=False, device=DEV, dtype=torch.bfloat16)}


@pytest.fixture(params=PROJECTIONS)
def projection(request):
    return PROJECTIONS[request.param]()


def _linear_of(m):
    """torch's own layer on the same weight."""
    lin = torch.nn.Linear(m.in_features, m.out_features, bias=False, device="meta")
    lin.weight = m.weight
    return lin


def _normal(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).bfloat16().to(DEV)


def _near(a, b):
    # two roundings to bfloat16 of nearly the same float32 sums
    return a.shape == b.shape and a.dtype == b.dtype and (a - b).float().norm() <= 2 ** -7 * b.float().norm()


def test_a_gradient_keeps_its_tangent(projection):
    """Forward mode entered after the forward call: the vector-Jacobian product is linear in dy, and so is its tangent."""
    x, dy, t = _normal(0, B, S, H * dh).requires_grad_(), _normal(1, B, S, projection.out_features), _normal(2, B, S, projection.out_features)
    got = []
    for m in (projection, _linear_of(projection)):
        y = m(x)
        with forward_ad.dual_level():
            grads = torch.autograd.grad(y, [x, m.weight], forward_ad.make_dual(dy, t))
            got.append([d for g in grads for d in forward_ad.unpack_dual(g)])
    assert all(d is not None for ds in got for d in ds)
    assert all(_near(a, b) for a, b in zip(*got))


def test_the_block_s_last_weight_keeps_its_gradient_s_tangent():
    layer, x, dY, t = _layer(), _normal(0, B, S, H * dh).requires_grad_(), _normal(1, B, S, H * dh), _normal(2, B, S, H * dh)
    y = layer(x)
    with forward_ad.dual_level():
        g, = torch.autograd.grad(y, [layer.w_self_2.weight], forward_ad.make_dual(dY, t), retain_graph=True)
        g = forward_ad.unpack_dual(g)
    want, = torch.autograd.grad(y, [layer.w_self_2.weight], t)
    assert g.tangent is not None and _near(g.tangent, want)


def test_gradients_in_batches(projection):
    x, dys = _normal(0, B, S, H * dh).requires_grad_(), _normal(1, 3, B, S, projection.out_features)
    y = projection(x)
    got = torch.autograd.grad(y, [x, projection.weight], dys, is_grads_batched=True, retain_graph=True)
    for i, dy in enumerate(dys):
        assert all(_near(a[i], b) for a, b in zip(got, torch.autograd.grad(y, [x, projection.weight], dy, retain_graph=True)))


class Seen(torch.Tensor):
    """Records what is dispatched on it; `Wrapper` has no memory of its own, `Memory` has."""
    __torch_function__ = torch._C._disabled_torch_function_impl
    names = []

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        Seen.names.append(str(func))
        tree = torch.utils._pytree
        plain = tree.tree_map_only(Seen, lambda t: t.plain, (args, kwargs or {}))
        return tree.tree_map_only(torch.Tensor, cls.of, func(*plain[0], **plain[1]))


class Wrapper(Seen):
    @staticmethod
    def of(t):
        r = torch.Tensor._make_wrapper_subclass(Wrapper, t.shape, strides=t.stride(), dtype=t.dtype, device=t.device,
                                                requires_grad=t.requires_grad)
        r.plain = t.detach()
        return r


class Memory(Seen):
    @staticmethod
    def of(t):
        r = torch.Tensor._make_subclass(Memory, t.detach(), t.requires_grad)
        r.plain = t.detach()
        return r


@pytest.mark.parametrize("cls", [Wrapper, Memory])
@pytest.mark.parametrize("where", ["x", "weight", "dy"])
def test_code_of_a_tensor_runs(projection, cls, where):
    x, dy = _normal(0, B, S, H * dh).requires_grad_(), _normal(1, B, S, projection.out_features)
    want = [projection(x)]
    want += torch.autograd.grad(want[0], [x, projection.weight], dy)
    if where == "x":
        x = cls.of(x)
    if where == "weight":
        projection.weight = torch.nn.Parameter(cls.of(projection.weight))
    Seen.names.clear()
    y = projection(x)
    assert where == "dy" or any("mm" in n for n in Seen.names) and isinstance(y, cls)
    Seen.names.clear()
    got = [y, *torch.autograd.grad(y, [x, projection.weight], cls.of(dy) if where == "dy" or isinstance(y, cls) else dy)]
    assert sum("mm" in n for n in Seen.names) == 2 and all(isinstance(t, cls) for t in got[1:])
    with torch.no_grad():
        assert all(_near(getattr(a, "plain", a), b) for a, b in zip(got, want))


def test_fake_tensors(projection):
    from torch._subclasses.fake_tensor import FakeTensor, FakeTensorMode
    mode = FakeTensorMode(allow_non_fake_inputs=True)
    x = mode.from_tensor(_normal(0, B, S, H * dh)).requires_grad_()
    with warnings.catch_warnings():
        warnings.filterwarnings("error", message=".*data.pointer")
        for inside in (False, True):
            with mode if inside else torch.enable_grad():
                y = projection(x)
                dx, dw = torch.autograd.grad(y, [x, projection.weight], torch.ones_like(y))
            assert all(type(t) is FakeTensor for t in (y, dx, dw)), inside
            assert y.shape == (B, S, projection.out_features) and dx.shape == x.shape and dw.shape == projection.weight.shape
