"""The native nodes' other callers: a trace, forward mode, functorch, second derivatives, captured graphs, pickled modules and
parameters inside flat buffers meet what a torch.autograd.Function and plain tensors give them."""
import copy
import io

import pytest
import torch

from flashmhf_amd import FlashFFNMoE, FlashMLP, FlashMLPMoE, MHFFNDecoder, MHFFNLayer
from flashmhf_amd.head_gate import head_norm_gate
from flashmhf_amd.mhffn_layer import CausalSelfAttention

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
B, S, H, dh, E, de = 2, 24, 2, 64, 3, 32


def _op_inputs(seed=0, single=False):
    g = torch.Generator().manual_seed(seed)
    Q = torch.randn(B, H, S, dh, generator=g).bfloat16()
    W = [(torch.randn(*((H, de) if single else (H, E, de)), dh, generator=g) * dh ** -0.5).bfloat16() for _ in range(3)]
    R = [] if single else [torch.softmax(torch.randn(B, H, S, E, generator=g), -1)]
    return [t.to(DEV) for t in (Q, *W, *R)]


def _layer(**kw):
    torch.manual_seed(0)
    return MHFFNLayer(H * dh, H, E, de, apply_rmsnorm=True, **kw).to(DEV).to(torch.bfloat16)


def _x(seed, **kw):
    return torch.randn(B, S, H * dh, generator=torch.Generator().manual_seed(seed)).bfloat16().to(DEV).requires_grad_(kw.get("grad", False))


@pytest.mark.parametrize("op,single", [(FlashMLPMoE(), False), (FlashMLPMoE(one_part=True), False), (FlashFFNMoE(), False), (FlashMLP(), True)])
def test_operator_under_trace_and_transforms(op, single):
    first, other = _op_inputs(0, single), _op_inputs(1, single)
    for grad in (False, True):
        traced = torch.jit.trace(op, (first[0], *(t.requires_grad_(grad) for t in first[1:])), check_trace=False)
        assert torch.equal(traced(*other), op(*other))      # not the constant of the first call
    with pytest.raises(Exception), torch.autograd.forward_ad.dual_level():
        op(torch.autograd.forward_ad.make_dual(first[0], torch.ones_like(first[0])), *first[1:])
    with pytest.raises(RuntimeError):
        torch.func.vmap(op)(*(torch.stack([t, t]) for t in first))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda q: op(q, *first[1:]).float().sum())(first[0])


@pytest.mark.parametrize("make", [_layer, lambda: CausalSelfAttention(H * dh, H).to(DEV).to(torch.bfloat16)])
def test_modules_under_trace(make):
    m = make()
    traced = torch.jit.trace(m, (_x(0),), check_trace=False)
    assert torch.equal(traced(_x(1)), m(_x(1)))


def test_layer_refuses_forward_mode():
    with pytest.raises(Exception), torch.autograd.forward_ad.dual_level():
        _layer()(torch.autograd.forward_ad.make_dual(_x(0), _x(1)))


def test_second_derivative_of_the_block_is_the_stepwise_one():
    layer, x, dY = _layer(), _x(0, grad=True), _x(1)
    out = []
    for stepwise in (False, True):
        if stepwise:
            layer.w_self.register_forward_hook(lambda *a: None)
        dw2, = torch.autograd.grad(layer(x), [layer.w_self_2.weight], dY, create_graph=True)
        out.append(torch.autograd.grad(dw2, [x], torch.ones_like(dw2))[0])
    assert torch.equal(*out)


@pytest.mark.parametrize("frozen", [(), ("w_self.weight",), ("w_self_2.weight", "K")])
def test_every_second_derivative_of_the_block_is_the_stepwise_one(frozen):
    """All first gradients under create_graph, and what they hand back to every tensor."""
    layer, x, dY = _layer(), _x(0, grad=True), _x(1, grad=True)
    params = {n: p.requires_grad_(n not in frozen) for n, p in layer.named_parameters()}
    leaves = [x, *(p for n, p in params.items() if n not in frozen)]
    out = []
    for stepwise in (False, True):
        if stepwise:
            layer.w_self.register_forward_hook(lambda *a: None)
        first = torch.autograd.grad(layer(x), leaves, dY, create_graph=True)
        loss = sum(g.float().square().mean() for g in first if g.requires_grad)
        out.append([*first, *torch.autograd.grad(loss, [*leaves, dY], allow_unused=True)])
    for i, (a, b) in enumerate(zip(*out)):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b)), i


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_parameters_at_any_place_of_a_flat_buffer(dtype):
    x4 = _x(0).view(B, S, H, dh)
    wn, router = torch.rand(H, dh, device=DEV).to(dtype) + 0.5, torch.randn(H, dh, E, device=DEV).to(dtype) * 0.1
    flat = torch.cat([wn.new_zeros(1), wn.flatten(), router.flatten()])
    views = [flat[1:1 + wn.numel()].view_as(wn).requires_grad_(), flat[1 + wn.numel():].view_as(router).requires_grad_()]
    results = []
    for ps in ([wn.requires_grad_(), router.requires_grad_()], views):
        Q, R = head_norm_gate(x4, *ps)
        results.append([Q, R, *torch.autograd.grad([Q, R], ps, [torch.ones_like(Q), torch.ones_like(R) * 0.5])])
    assert all(torch.equal(a, b) for a, b in zip(*results))



def test_attention_takes_tables_of_other_forms():
    attn = CausalSelfAttention(H * dh, H).to(DEV).to(torch.bfloat16)
    cos, sin = (torch.randn(S, dh, device=DEV).bfloat16() for _ in range(2))
    want = attn(_x(0), rope=(cos, sin))
    assert torch.equal(attn(_x(0), rope=(cos.view(1, S, dh), sin.view(1, S, dh))), want)
    odd = torch.empty(2 * S * dh + 1, device=DEV).bfloat16()[1:].view(2, S, dh)
    odd[0], odd[1] = cos, sin
    assert torch.equal(attn(_x(0), rope=tuple(odd)), want)
    cos.requires_grad_()
    assert torch.autograd.grad(attn(_x(0), rope=(cos, sin)).sum(), cos)[0].abs().sum() > 0


def _decoder():
    torch.manual_seed(0)
    return MHFFNDecoder(64, H * dh, 2, H, H, E, de).to(DEV).to(torch.bfloat16)


def test_captured_decoder_outlives_the_kept_tables():
    m = _decoder()
    ids = torch.randint(0, 64, (B, S), device=DEV)
    st = torch.cuda.Stream()
    with torch.no_grad(), torch.cuda.stream(st):
        want = m(ids)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            got = m(ids)
        for k in range(1, 4):
            m(ids[:, :S - k])                                   # another length takes the place of the kept tables
            junk = [torch.full((S, dh), 7.0, device=DEV).bfloat16() for _ in range(64)]
            g.replay()
            st.synchronize()
            assert torch.equal(got, want)
            del junk


def test_copies_and_files_go_without_the_tables():
    m = _decoder()
    ids = torch.randint(0, 64, (B, S), device=DEV)
    with torch.no_grad():
        want = m(ids)
        f = io.BytesIO()
        torch.save(m, f)
        f.seek(0)
        for other in (copy.deepcopy(m), torch.load(f, weights_only=False)):
            assert "_rope_kept" not in other.__dict__
            assert torch.equal(other(ids), want)


def test_operator_saved_before_it_had_a_choice():
    op = FlashMLPMoE()
    del op.__dict__["one_part"]
    ins = _op_inputs()
    assert torch.equal(op(*ins), FlashMLPMoE()(*ins))
