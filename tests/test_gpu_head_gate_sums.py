"""Head prologue backward where a wave takes several tiles and many workgroups' sums meet (more than 2,048 tiles of 32 tokens,
ragged ends, several batches), for float32 and bfloat16 parameters: against torch autograd on the same inputs in float32, and
twice for the same bits."""
import pytest
import torch

from oracle import mhffn_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,H,dh,E,norm", [(3, 11003, 8, 64, 5, True), (1, 33000, 4, 96, 32, True), (2, 20001, 4, 128, 22, True),
                                             (2, 17000, 4, 128, 3, False), (1, 9000, 4, 64, 33, True)])
@pytest.mark.parametrize("wn_bf16,wr_bf16", [(True, False), (False, True)])
def test_many_tiles(B, S, H, dh, E, norm, wn_bf16, wr_bf16):
    from flashmhf_amd.head_gate import head_norm_gate
    print(f"case B={B} S={S} H={H} dh={dh} E={E} norm={norm} {wn_bf16} {wr_bf16}", flush=True)
    dev = "cuda:0"
    g = torch.Generator(device=dev).manual_seed(S)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)
    x = r(B, S, H, dh).bfloat16().requires_grad_(True)
    wn = (1 + 0.1 * r(H, dh)).to(torch.bfloat16 if wn_bf16 else torch.float32).requires_grad_(True) if norm else None
    wr = (0.1 * r(H, dh, E)).to(torch.bfloat16 if wr_bf16 else torch.float32).requires_grad_(True)
    dQ, dR = r(B, S, H, dh).bfloat16().transpose(1, 2), r(B, H, S, E)
    leaves = [x, wr] + ([wn] if norm else [])
    got, again = (torch.autograd.grad(head_norm_gate(x, wn, wr, 1e-6), leaves, [dQ, dR]) for _ in range(2))
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    xf, wrf = x.detach().float().requires_grad_(True), wr.detach().float().requires_grad_(True)
    wnf = wn.detach().float().requires_grad_(True) if norm else None
    q = torch.nn.functional.rms_norm(xf, (dh,), None, 1e-6) * wnf if norm else xf
    z = torch.matmul(q.transpose(1, 2).contiguous(), wrf)
    s = z.sigmoid()
    R = s / s.sum(-1, keepdim=True).clamp(min=1e-20)
    ref = torch.autograd.grad([q.transpose(1, 2), R], [xf, wrf] + ([wnf] if norm else []), [dQ.float(), dR])
    for name, a, b in zip(("dx", "d_router", "d_norm"), got, ref):
        m = orc.error_metrics(a.float().cpu(), b.cpu())
        print(name, m, flush=True)
        assert m["norm_max"] <= 2e-2 and m["mean_rel"] <= 1e-2, (name, m)
