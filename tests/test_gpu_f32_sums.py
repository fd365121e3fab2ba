"""float32: the pass that adds up the parts counts tiles and heads as the kernels that left them (padded grids of 128-row tiles and others, a
last tile of few rows, rows of d_h that end inside a workgroup), and dK/dU/dV's workgroups with the head fastest and, in slices, not."""
import pytest
import torch

from flashmhf_amd import _capi
from tests.helpers import make_inputs

DEV = "cuda:0"

# B, H, S, dh, E, de, Hk; padded grid, several token slices
CASES = [((1, 3, 129, 40, 5, 37, 3), True, True), ((2, 10, 150, 72, 3, 64, 5), False, True), ((1, 4, 300, 96, 6, 33, 2), True, True),
         ((1, 1, 40, 8, 70, 31, 1), False, False), ((1, 8, 32, 64, 10, 224, 8), False, False), ((1, 33, 70, 24, 8, 65, 33), False, False)]


@pytest.mark.parametrize("dims,padded,slices", CASES)
def test_what_the_cases_cover(dims, padded, slices):
    B, H, S, dh, E, de, Hk = dims
    p = _capi.launch_plan(_capi.Dims(B, H, Hk, S, dh, E, de), _capi.DTYPE_F32)
    tiles, parts = -(-B * S * H // Hk // 128) * Hk, p.fwd_parts
    assert parts > 1 and p.dqdr_parts > 1 and (p.dkdudv_slices > 1) is slices
    assert bool(_capi.launch_forms(_capi.Dims(B, H, Hk, S, dh, E, de), _capi.DTYPE_F32) & _capi.FORM_FWD_PADDED) is padded
    assert not padded or (tiles % 8 != 0 and tiles <= 24 and -(-tiles // 8) * parts <= 32 * -(-tiles * parts // 256))


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [c[0] for c in CASES])
def test_sums_match_the_oracle(dims):
    from flashmhf_amd import mhffn_backward, mhffn_forward
    from oracle import mhffn_oracle as orc
    print("case", dims, flush=True)
    B, H, S, dh, E, de, Hk = dims
    ins = make_inputs(B, H, S, dh, E, de, Hk, seed=17)
    dev = [t.to(DEV) for t in ins]
    got = (mhffn_forward(*dev[:5]), *mhffn_backward(*dev, grad_w_dtype=torch.float32))
    torch.cuda.synchronize()
    ref = (orc.mhffn_forward(*ins[:5], compute_dtype=torch.float64), *orc.mhffn_backward(*ins, compute_dtype=torch.float64))
    for name, a, r in zip(("O", "dQ", "dK", "dU", "dV", "dR"), got, ref):
        err = (a.double().cpu() - r).abs().max().item()      # (the bar of the other float32 cases with parts and slices)
        assert err <= 1e-5 * max(1.0, r.abs().max().item()), (name, dims, err)
