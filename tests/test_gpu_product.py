"""The block's projections through the C ABI at the sizes where their tiles, stages and waves begin and end, against the same sums
in float64.  A result is at most one rounding to bfloat16 (2^-8 of its value, half an ulp 2^-9) and the float32 sums' error (K terms,
each 2^-24 of the absolute terms' sum at worst) away from it."""
import pytest
import torch

from flashmhf_amd import _capi

pytestmark = pytest.mark.gpu
NT, NN, TN = _capi.PRODUCT_NT, _capi.PRODUCT_NN, _capi.PRODUCT_TN


def _case(form, M, N, K, in_order, seed=0):
    dev = "cuda:0"
    g = torch.Generator(device=dev).manual_seed(seed)
    shapes = {NT: ((M, K), (N, K)), NN: ((M, K), (K, N)), TN: ((K, M), (K, N))}[form]
    a, b = (torch.randn(*s, generator=g, device=dev).bfloat16() for s in shapes)
    # (behind the result and the operands lies what must not be touched or read)
    out = torch.full((M * N + 64,), 7.0, device=dev, dtype=torch.bfloat16)
    pad = [torch.cat([t.reshape(-1), torch.full((64,), float("nan"), device=dev, dtype=torch.bfloat16)]) for t in (a, b)]
    rc = _capi.lib().mhffn_product(form, in_order, pad[0].data_ptr(), pad[1].data_ptr(), out.data_ptr(), M, N, K,
                                   torch.cuda.current_stream().cuda_stream)
    assert rc == _capi.OK
    assert (out[M * N:] == 7.0).all()
    x, y = (t.double() for t in (a, b))
    if form == NT:
        y = y.t()
    if form == TN:
        x = x.t()
    ref, mag = x.contiguous() @ y.contiguous(), x.abs().contiguous() @ y.abs().contiguous()
    err = (out[:M * N].view(M, N).double() - ref).abs()
    assert (err <= ref.abs() * 2 ** -8 + mag * K * 2 ** -24).all(), (form, M, N, K, err.max().item())


SIZES = [(8, 8), (24, 40), (72, 96), (136, 128), (264, 192), (496, 1000), (1000, 1000), (2040, 1000), (2056, 1544), (4104, 2056)]


# rows x columns of every tile, with edges inside a tile, one and several rounds of workgroups
@pytest.mark.parametrize("form,in_order", [(NT, 0), (NT, 1), (NN, 0), (TN, 0)])
@pytest.mark.parametrize("M,N", SIZES)
# one chunk of 64 and less, the stages' edges, fewer chunks than waves, more stages than the ring holds
@pytest.mark.parametrize("K", [8, 64, 72, 136, 512, 1096])
def test_products(form, in_order, M, N, K):
    print(f"form {form} M={M} N={N} K={K} in_order={in_order}", flush=True)
    _case(form, M, N, K, in_order, seed=M + N + K)


@pytest.mark.parametrize("form,M,N,K", [(NT, 1, 768, 768), (NT, 17, 2048, 2048), (NT, 733, 768, 768), (NN, 1, 64, 64), (NN, 37, 96, 96),
                                        (TN, 64, 64, 1), (TN, 96, 96, 37), (TN, 768, 768, 1025)])
def test_products_of_odd_token_counts(form, M, N, K):
    for in_order in (0, 1):
        _case(form, M, N, K, in_order, seed=K)


def test_every_tile_is_one_of_the_cases():
    tile = _capi.lib().mhffn_product_tile
    tiles = {(form, o): {divmod(tile(form, o, M, N, 512), 65536) for M, N in SIZES} for form in (NT, NN, TN) for o in (0, 1)}
    large = {(64, 64), (128, 64), (128, 128)}
    assert tiles == {(NT, 0): large | {(32, 32), (64, 32)}, (NT, 1): large | {(32, 64)}, **{(f, o): large for f in (NN, TN) for o in (0, 1)}}
    assert not tile(NT, 0, 8, 8, 12) and not tile(TN, 0, 12, 8, 8)


@pytest.mark.parametrize("M,N,K", [(17, 192, 192), (64, 1024, 1024), (300, 768, 768), (512, 3072, 1024), (1000, 1024, 1024), (2048, 768, 768)])
def test_sums_in_order_have_the_library_s_bits(M, N, K):
    """OrderedProjection, values and gradients, against nn.Linear."""
    from flashmhf_amd.mhffn_layer import OrderedProjection
    dev = "cuda:0"
    torch.manual_seed(M)
    own = OrderedProjection(K, N, bias=False, device=dev, dtype=torch.bfloat16)
    lib = torch.nn.Linear(K, N, bias=False, device=dev, dtype=torch.bfloat16)
    lib.load_state_dict(own.state_dict())
    x, dy = torch.randn(M, K, device=dev).bfloat16(), torch.randn(M, N, device=dev).bfloat16()
    results = []
    for m in (own, lib):
        xi = x.clone().requires_grad_(True)
        y = m(xi)
        results.append((y, *torch.autograd.grad(y, [xi, m.weight], dy)))
    for a, b in zip(*results):
        assert torch.equal(a, b)


# sizes at which the library sums in another order: nothing but its own products has its bits
@pytest.mark.parametrize("M,N,K", [(17, 1024, 1024), (24, 768, 768), (31, 2048, 768), (128, 1024, 4096), (96, 1280, 1280), (80, 1536, 1536),
                                   (64, 2048, 2048), (144, 1792, 1792)])
def test_ordered_projections_of_few_rows_have_the_library_s_bits(M, N, K):
    test_sums_in_order_have_the_library_s_bits(M, N, K)


@pytest.mark.parametrize("T", [1, 16, 300, 2048])
def test_the_block_projects_as_a_linear_layer_does(T):
    """A captured graph of the block, replayed with the program's own work between, gives what an eager call gives, and a dispatch
    mode still sees the products."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from flashmhf_amd import MHFFNLayer
    dev = "cuda:0"
    torch.manual_seed(T)
    with torch.device(dev):
        m = MHFFNLayer(512, 4, 3, 64, apply_rmsnorm=True).to(torch.bfloat16).requires_grad_(False)
    x = torch.randn(1, T, 512, device=dev).bfloat16()
    want = m(x)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        got = m(x)
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        m(torch.randn_like(x))

    class Seen(TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))
    with Seen() as seen:
        m(x)
    assert sum("mm" in n or "linear" in n for n in seen.names) == 2


@pytest.mark.parametrize("trained", [("x",), ("w",), ("x", "w")])
@pytest.mark.parametrize("T", [1, 70])
def test_projection_is_a_linear_layer(T, trained):
    """Values and gradients of any order against torch's linear layer, in what is kept for the backward no more than it keeps."""
    from flashmhf_amd.mhffn_layer import Projection
    dev = "cuda:0"
    torch.manual_seed(T)
    own = Projection(192, 320, bias=False, device=dev, dtype=torch.bfloat16)
    lib = torch.nn.Linear(192, 320, bias=False, device=dev, dtype=torch.bfloat16)
    lib.load_state_dict(own.state_dict())
    x, dy, v = (torch.randn(*s, device=dev).bfloat16() for s in ((2, T, 192), (2, T, 320), (2, T, 192)))
    results = []
    for m in (own, lib):
        m.weight.requires_grad_("w" in trained)
        xi = x.clone().requires_grad_("x" in trained)
        leaves = [t for n, t in (("x", xi), ("w", m.weight)) if n in trained]
        dyi = dy.clone().requires_grad_(True)
        y = m(xi)
        grads = torch.autograd.grad(y, leaves, dyi, create_graph=True)
        second = torch.autograd.grad(sum((g.float() ** 2).sum() for g in grads), [dyi])
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
            plain = torch.autograd.grad(m(xi), leaves, dy)
        names = {e.key: e.count for e in prof.key_averages()}
        results.append((y, *grads, *second, *plain))
        assert (names.get("mhffn::product", 0), names.get("aten::mm", 0)) == ((1 + len(leaves), 0) if m is own else (0, 1 + len(leaves)))
    for a, b in zip(*results):
        assert a.shape == b.shape and a.dtype == b.dtype
        # two roundings to bfloat16 of nearly the same sums; the second derivative has rounded factors
        assert (a - b).float().norm() <= 2 ** -7 * b.float().norm()


@pytest.mark.parametrize("by", ["frozen", "named"])
@pytest.mark.parametrize("trained,products", [({"K"}, 3), ({"w_self.weight"}, 4), ({"w_self_2.weight"}, 3), ({"router", "w_self_2.weight"}, 4)])
def test_products_that_nobody_asks_for_are_not_taken(trained, products, by):
    """Forward two; backward dO for anything in front of the operator, dw for a projection that is asked for; with steps as well."""
    from flashmhf_amd import MHFFNLayer
    dev = "cuda:0"
    torch.manual_seed(0)
    layer = MHFFNLayer(128, 2, 3, 32, apply_rmsnorm=True).to(dev).to(torch.bfloat16)
    for name, p in layer.named_parameters():
        p.requires_grad_(by == "named" or name in trained)
    x = torch.randn(2, 24, 128, device=dev).bfloat16()
    asked = [p for name, p in layer.named_parameters() if name in trained]
    for stepwise in (False, True):
        if stepwise:
            layer.w_self.register_forward_hook(lambda *a: None)
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
            torch.autograd.grad(layer(x), asked, torch.ones_like(x))
        counts = {e.key: e.count for e in prof.key_averages()}
        assert (counts.get("mhffn::product"), counts.get("aten::mm", 0)) == (products, 0), stepwise


# (own products of: y, dx, dw; the others are the library's)
@pytest.mark.parametrize("T,hidden,own", [(8, 320, 3), (8, 1024, 2), (32, 1024, 3), (63, 2048, 2), (64, 2048, 3), (160, 3072, 1)])
def test_few_rows_and_long_sums_take_the_faster_product(T, hidden, own):
    from flashmhf_amd.mhffn_layer import Projection
    dev = "cuda:0"
    torch.manual_seed(T)
    m = Projection(hidden, hidden, bias=False, device=dev, dtype=torch.bfloat16)
    x, dy = (torch.randn(T, hidden, device=dev).bfloat16() for _ in range(2))
    x.requires_grad_()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        y = m(x)
        dx, dw = torch.autograd.grad(y, [x, m.weight], dy)
    names = {e.key: e.count for e in prof.key_averages()}
    assert (names.get("mhffn::product", 0), names.get("aten::mm", 0)) == (own, 3 - own)
    a, b, w = (t.detach().double() for t in (x, dy, m.weight))
    for got, p, q, K in ((y, a, w.t().contiguous(), hidden), (dx, b, w, hidden), (dw, b.t().contiguous(), a, T)):
        ref, mag = p @ q, p.abs() @ q.abs()
        assert ((got.double() - ref).abs() <= ref.abs() * 2 ** -8 + mag * K * 2 ** -24).all()


@pytest.mark.parametrize("B,S", [(1, 24), (1, 300), (3, 200)])
def test_a_decoder_of_linear_layers_has_the_same_bits(B, S):
    """The decoder's own projections against torch's layers throughout, loss and every gradient."""
    from flashmhf_amd import MHFFNDecoder
    dev = "cuda:0"
    ids = torch.randint(0, 512, (B, S), device=dev, generator=torch.Generator(device=dev).manual_seed(S))
    results = []
    for kw in ({}, {"linear": torch.nn.Linear}):
        torch.manual_seed(0)
        with torch.device(dev):
            m = MHFFNDecoder(512, 768, 2, 8, 8, 3, 64, **kw).to(torch.bfloat16)
        loss = m(ids, labels=ids)
        results.append((loss, *torch.autograd.grad(loss, list(m.parameters()))))
    for a, b in zip(*results):
        assert torch.equal(a, b)


# (y = x w^T of M x K by N x K.)  Edges of every tile, one workgroup to several rounds, sums shorter than a stage and longer than the ring
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (1, 64, 64), (37, 72, 40), (64, 1096, 264), (129, 136, 1000), (300, 768, 768), (512, 1024, 1024),
                                   (700, 768, 768), (733, 1032, 1032), (1024, 1024, 1024), (1025, 768, 768), (1500, 1024, 1024),
                                   (2056, 1544, 520), (4104, 768, 768), (512, 8192, 264), (700, 2048, 2048), (512, 3072, 1024), (512, 2048, 2048)])
def test_a_pair_has_the_bits_of_its_products(M, N, K):
    dev = "cuda:0"
    print(f"M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    nan = torch.full((64,), float("nan"), device=dev, dtype=torch.bfloat16)
    # (behind the operands lies what must not be read, behind the results what must not be touched)
    dy, w, x = (torch.cat([torch.randn(n, generator=g, device=dev).bfloat16(), nan]) for n in (M * N, N * K, M * K))
    out = [torch.full((n + 64,), 7.0, device=dev, dtype=torch.bfloat16) for n in (M * K, N * K, M * K, N * K)]
    L, st = _capi.lib(), torch.cuda.current_stream().cuda_stream
    assert L.mhffn_product_pair(dy.data_ptr(), w.data_ptr(), x.data_ptr(), out[0].data_ptr(), out[1].data_ptr(), M, N, K, st) == _capi.OK
    assert L.mhffn_product(NN, 1, dy.data_ptr(), w.data_ptr(), out[2].data_ptr(), M, K, N, st) == _capi.OK
    assert L.mhffn_product(TN, 1, dy.data_ptr(), x.data_ptr(), out[3].data_ptr(), N, K, M, st) == _capi.OK
    assert torch.equal(out[0], out[2]) and torch.equal(out[1], out[3]) and all((o[-64:] == 7.0).all() for o in out)
    assert torch.isfinite(out[0]).all() and torch.isfinite(out[1]).all()
