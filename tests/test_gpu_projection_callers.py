"""What meets the projections' own products as it meets torch's linear layer: forward mode in the backward alone."""
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
