"""Head prologue backward on both sides of the rule that picks four or eight waves per workgroup (1,024 tiles of 32 tokens over
all heads, up to 32 experts), with waves that have no tile: sums over tokens against float64, and dx, which depends on a token's own
row alone, bit for bit the same on both sides."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,H,dh,E", [(1, 2, 128, 1), (33, 3, 96, 32), (129, 2, 64, 17), (160, 1, 128, 32), (1000, 16, 96, 11),
                                      (8160, 4, 128, 22), (8161, 4, 128, 22), (8160, 4, 64, 5), (8192, 4, 64, 5), (8170, 4, 96, 8)])
def test_either_number_of_waves(S, H, dh, E):
    from flashmhf_amd import _capi
    print(f"case S={S} H={H} dh={dh} E={E}", flush=True)
    dev = "cuda:0"
    g = torch.Generator(device=dev).manual_seed(S + dh)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)
    n = 8200      # rows of the inputs, of which a call takes the first S
    X, DQ, DR = r(n, H, dh).bfloat16(), r(n, H, dh).bfloat16(), r(n, H, E)
    wn, wr = 1 + 0.1 * r(H, dh), 0.1 * r(H, dh, E)

    def call(m):
        dQ, dR = DQ[:m].permute(1, 0, 2)[None], DR[:m].permute(1, 0, 2)[None].contiguous()
        return _capi.native().gate_backward(X[None, :m].contiguous(), wn, wr, 1e-6, dQ.contiguous(), dR)

    dx, dwn, dwr = call(S)
    assert torch.equal(dx[0], call(n)[0][0, :S])

    x, dq, dr = X[:S].double(), DQ[:S].double(), DR[:S].double()
    u = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
    y = (u * wn.double()).bfloat16().double()
    z = torch.stack([y[:, h] @ wr[h].double() for h in range(H)], 1)
    s = z.sigmoid()
    tot = s.sum(-1, keepdim=True)
    R = s / tot
    dz = (dr - (dr * R).sum(-1, keepdim=True)) / tot * s * (1 - s)
    # d_router: y exactly the kernel's except where a product lies on a rounding boundary (2^-8 of an element), dz rounded to bfloat16 (2^-9)
    for h in range(H):
        ref, mag = y[:, h].T @ dz[:, h], y[:, h].abs().T @ dz[:, h].abs()
        assert bool(((dwr[h].double() - ref).abs() <= 2.0 ** -7 * mag + 1e-6).all())
        # d_norm_weight: d = dQ + dy, dy from dz and the router rounded to bfloat16 (2^-9 each, and z's own error below that)
        dy, dmag = dz[:, h] @ wr[h].double().T, dz[:, h].abs() @ wr[h].double().abs().T
        d = dq[:, h] + dy
        err = ((2.0 ** -7 * dmag + 2.0 ** -20 * d.abs()) * u[:, h].abs()).sum(0)
        assert bool(((dwn[h].double() - (d * u[:, h]).sum(0)).abs() <= err + 1e-6).all())
