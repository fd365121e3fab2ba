"""Head prologue with rows moved whole through LDS (many tokens) against rows moved in half rows' pieces (few): the same arithmetic,
so Q, R and dx agree bit for bit, also where the last tile is not full; and the sums over tokens of backward launches whose waves take
one tile or several."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(B, S, H, dh, E, norm):
    g = torch.Generator(device=DEV).manual_seed(S + dh)
    x = torch.randn(B, S, H, dh, generator=g, device=DEV).bfloat16()
    wn = 1 + 0.1 * torch.randn(H, dh, generator=g, device=DEV) if norm else None
    return x, wn, 0.1 * torch.randn(H, dh, E, generator=g, device=DEV), g


# 1,536 tiles of 32 tokens over all heads and batches (from 1,024 on whole rows move): last tiles of 1, 31 and 32 rows
@pytest.mark.parametrize("B,S,H,dh,E,norm", [(1, 3041, 16, 128, 22, True), (2, 3071, 8, 96, 8, True), (4, 3072, 4, 64, 32, True),
                                             (1, 3050, 16, 128, 11, False), (1, 3041, 16, 96, 40, True)])
def test_forward(B, S, H, dh, E, norm):
    from flashmhf_amd.head_gate import head_norm_gate
    print(f"case B={B} S={S} H={H} dh={dh} E={E} norm={norm}", flush=True)
    assert B * H * ((S + 31) // 32) >= 1536
    x, wn, router, _ = _inputs(B, S, H, dh, E, norm)
    Q, R = head_norm_gate(x, wn, router, 1e-6)
    for b in range(B):
        for t in (0, 512, S - 500):      # (calls of 500 tokens: pieces)
            q, r = head_norm_gate(x[b:b + 1, t:t + 500].contiguous(), wn, router, 1e-6)
            assert torch.equal(Q[b, :, t:t + 500], q[0]) and torch.equal(R[b, :, t:t + 500], r[0])


# (32 and more experts, and 16 for heads below 128, stay with pieces: the cases above with 32 and 40)
@pytest.mark.parametrize("B,S,H,dh,E,norm", [(4, 3072, 4, 64, 31, True), (1, 3041, 16, 96, 17, True), (2, 3050, 8, 128, 16, True), (1, 6200, 8, 64, 8, False),
                                             (1, 3041, 16, 96, 16, True)])
def test_forward_around_the_experts_of_that_rule(B, S, H, dh, E, norm):
    test_forward(B, S, H, dh, E, norm)


# 8,192 tiles: four of them per wave, dx whole; 3,104 and 2,080: two per wave instead of a second round of workgroups
@pytest.mark.parametrize("B,S,H,dh,E,norm", [(1, 16353, 16, 128, 22, True), (2, 16384, 8, 96, 8, True), (1, 32767, 8, 64, 17, True),
                                             (1, 16360, 16, 128, 11, False), (1, 12390, 8, 128, 11, True), (5, 3300, 4, 64, 8, True)])
@pytest.mark.parametrize("token_major", [True, False])
def test_backward(B, S, H, dh, E, norm, token_major):
    from flashmhf_amd import _capi
    print(f"case B={B} S={S} H={H} dh={dh} E={E} norm={norm} token_major={token_major}", flush=True)
    x, wn, router, g = _inputs(B, S, H, dh, E, norm)
    dQ = torch.randn(B, S, H, dh, generator=g, device=DEV).bfloat16().transpose(1, 2)
    if not token_major:
        dQ = dQ.contiguous()
    dR = torch.randn(B, H, S, E, generator=g, device=DEV)
    back = _capi.native().gate_backward
    dx, dwn, dwr = back(x, wn, router, 1e-6, dQ, dR)
    sums = [torch.zeros_like(t, dtype=torch.float64) if t is not None else None for t in (dwn, dwr)]
    size = [torch.zeros_like(t) if t is not None else None for t in sums]
    for b in range(B):
        for t in range(0, S, 1000):
            cut = slice(t, min(t + 1000, S))
            dx1, dwn1, dwr1 = back(x[b:b + 1, cut].contiguous(), wn, router, 1e-6, dQ[b:b + 1, :, cut], dR[b:b + 1, :, cut].contiguous())
            assert torch.equal(dx[b, cut], dx1[0])
            for s, z, part in zip(sums, size, (dwn1, dwr1)):
                if s is not None:
                    s += part
                    z += part.abs()
    # float32 sums of the same terms in two orders: each off by at most 2^-24 of the terms' size per addition, of about 1,000 in a row
    for s, z, whole in zip(sums, size, (dwn, dwr)):
        if s is not None:
            assert bool(((whole.double() - s).abs() <= 2.0 ** -14 * (z + z.mean())).all())
