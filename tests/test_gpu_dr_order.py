"""dQ and dR of 32-row tiles, whose four waves add their blocks to dR one after the other: experts of one to seven blocks, so that they begin
and end at every wave, last trips of one to four blocks, one trip and many, against the 256-row tiles' results for the same rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("E,de", [(1, 32), (2, 32), (64, 32), (7, 64), (5, 96), (3, 128), (9, 160), (3, 224)])
def test_rows_have_the_same_sums_in_small_and_large_tiles(dh, E, de):
    from flashmhf_amd import mhffn_backward
    print("case", dh, E, de, flush=True)
    H, S = 16, 4000
    g = torch.Generator(device=DEV).manual_seed(dh + E)
    r = lambda *s, scale=1.0: (torch.randn(*s, generator=g, device=DEV) * scale).bfloat16()
    Q, dO = r(1, H, S, dh), r(1, H, S, dh)
    K, U, V = (r(H, E, de, dh, scale=dh ** -0.5) for _ in range(3))
    R = torch.rand(1, H, S, E, generator=g, device=DEV)
    all_rows = mhffn_backward(Q, K, U, V, R, dO, one_part=True)
    for n in (1, 33):
        few = slice(S - n, S)
        q, rr, d = (t[:, :, few].contiguous() for t in (Q, R, dO))
        got = mhffn_backward(q, K, U, V, rr, d, one_part=True)
        assert torch.equal(got[0], all_rows[0][:, :, few])
        assert torch.equal(got[4], all_rows[4][:, :, few])
