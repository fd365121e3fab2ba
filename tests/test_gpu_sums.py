"""The passes that add up parts and token slices count their workgroups as the kernels that left them did (whole_xcds in
csrc/mhffn_common.hpp): numbers of tiles that are padded and that are not, a last tile of few rows, heads that are no power of two, as many
experts as a part's dR has columns, columns of weights that end inside a workgroup."""
import pytest
import torch

from flashmhf_amd import _capi
from tests.helpers import assert_bf16_parity, make_inputs

DEV = "cuda:0"

# B, H, S, dh, E, de, Hk
CASES = [(1, 3, 129, 128, 9, 256, 3), (1, 5, 300, 96, 7, 160, 5), (2, 6, 700, 64, 12, 288, 3), (1, 1, 40, 64, 64, 32, 1), (1, 12, 300, 64, 7, 192, 12),
         (1, 8, 600, 128, 11, 352, 2), (1, 7, 520, 96, 5, 224, 7)]


def test_the_cases_cover_padded_grids_and_others():
    seen = {"fwd": set(), "dq": set(), "slices": set()}
    for B, H, S, dh, E, de, Hk in CASES:
        d = _capi.Dims(B, H, Hk, S, dh, E, de)
        p, forms = _capi.launch_plan(d, _capi.DTYPE_BF16), _capi.launch_forms(d, _capi.DTYPE_BF16)
        for name, height, parts, bit in (("fwd", p.fwd_tile_rows, p.fwd_parts, _capi.FORM_FWD_PADDED), ("dq", p.dqdr_tile_rows, p.dqdr_parts, _capi.FORM_DQDR_PADDED)):
            assert parts > 1
            tiles = -(-B * S * H // Hk // height) * Hk
            assert not forms & bit or (tiles % 8 != 0 and -(-tiles // 8) * parts <= 32 * -(-tiles * parts // 256))
            seen[name].add(bool(forms & bit))
        seen["slices"].add(p.dkdudv_slices > 1)
    assert all(s == {False, True} for s in seen.values())


# B, H, Hk, S, dh, E, de, padded: both sides of the lines (weights for 256-row tiles; what an XCD reads more for smaller ones)
@pytest.mark.parametrize("B,H,Hk,S,dh,E,de,fwd,dq", [(8, 8, 2, 1, 128, 11, 352, False, False), (1, 8, 2, 270, 96, 8, 256, True, True), (1, 6, 6, 39, 128, 16, 352, False, False),
                                                     (1, 6, 3, 1, 64, 4, 384, True, False), (2, 6, 6, 1600, 128, 16, 352, False, False), (4, 8, 4, 346, 128, 11, 352, False, False),
                                                     (8, 4, 2, 459, 64, 13, 256, True, True), (8, 8, 8, 64, 128, 11, 352, False, False), (8, 8, 2, 171, 128, 11, 352, False, False), (1, 8, 8, 2048, 128, 11, 352, False, False)])
def test_grids_are_padded_where_the_sums_save_more(B, H, Hk, S, dh, E, de, fwd, dq):
    forms = _capi.launch_forms(_capi.Dims(B, H, Hk, S, dh, E, de), _capi.DTYPE_BF16)
    assert (bool(forms & _capi.FORM_FWD_PADDED), bool(forms & _capi.FORM_DQDR_PADDED)) == (fwd, dq)


@pytest.mark.gpu
@pytest.mark.parametrize("dims", CASES)
@pytest.mark.parametrize("weights", [torch.bfloat16, torch.float32])
def test_sums_match_the_oracle(dims, weights):
    from flashmhf_amd import mhffn_backward, mhffn_forward
    from oracle import mhffn_oracle as orc
    print("case", dims, weights, flush=True)
    B, H, S, dh, E, de, Hk = dims
    ins = make_inputs(B, H, S, dh, E, de, Hk, seed=13, dtype=torch.bfloat16)
    dev = [t.to(DEV) for t in ins]
    got = (mhffn_forward(*dev[:5]), *mhffn_backward(*dev, grad_w_dtype=weights))
    torch.cuda.synchronize()
    ref = (orc.mhffn_forward(*ins[:5], compute_dtype=torch.float64), *orc.mhffn_backward(*ins, compute_dtype=torch.float64))
    for name, a, r in zip(("O", "dQ", "dK", "dU", "dV", "dR"), got, ref):
        assert_bf16_parity(name, a.float().cpu(), r, (dims, weights))
