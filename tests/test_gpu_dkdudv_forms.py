"""dK/dU/dV in each of its forms: one wave a block of rows or two (TokenHalves in csrc/mhffn_bwd.hip), one token slice or several, sequences of whole
tiles or not, for every head width.  The form is asserted without a GPU, so that a case whose form is no longer picked for it fails instead of testing another one."""
import pytest
import torch

from flashmhf_amd import _capi
from tests.helpers import assert_bf16_parity, make_inputs

DEV = "cuda:0"

# d_h: (B, H, S, E, de, Hk), two waves a block, token slices
ONE_SLICE = [((1, 32, 96, 4, 256, 32), False, 1), ((1, 32, 70, 4, 256, 32), False, 1), ((2, 2, 96, 3, 64, 2), True, 1), ((1, 6, 90, 5, 96, 3), True, 1)]
CASES = {
    64: [*ONE_SLICE, ((3, 6, 320, 11, 128, 6), False, 3), ((8, 12, 33, 11, 128, 6), False, 3), ((3, 4, 256, 3, 96, 2), True, 6), ((3, 6, 250, 3, 96, 3), True, 6)],
    96: [*ONE_SLICE, ((3, 6, 512, 11, 128, 6), False, 3), ((8, 24, 33, 11, 128, 6), False, 3), ((3, 4, 256, 3, 96, 2), True, 6), ((3, 6, 250, 3, 96, 3), True, 6)],
    128: [*ONE_SLICE, ((3, 8, 640, 11, 128, 4), False, 5), ((8, 16, 100, 11, 128, 4), False, 5), ((3, 4, 256, 3, 96, 2), True, 6), ((3, 6, 250, 3, 96, 3), True, 6)],
}
ALL = [(dh, *case) for dh, cases in CASES.items() for case in cases]


def _dims(dh, dims):
    B, H, S, E, de, Hk = dims
    return _capi.Dims(B, H, Hk, S, dh, E, de)


@pytest.mark.parametrize("dh,dims,halves,slices", ALL)
def test_the_case_runs_the_form_it_is_for(dh, dims, halves, slices):
    d = _dims(dh, dims)
    assert bool(_capi.launch_forms(d, _capi.DTYPE_BF16) & _capi.FORM_TOKEN_HALVES) is halves
    assert _capi.launch_plan(d, _capi.DTYPE_BF16).dkdudv_slices == slices


def test_the_cases_cover_every_form():
    for cases in CASES.values():
        assert len({(halves, slices > 1, dims[2] % 32 != 0) for dims, halves, slices in cases}) == 8


@pytest.mark.gpu
@pytest.mark.parametrize("dh,dims,halves,slices", ALL)
def test_gradients_match_the_oracle(dh, dims, halves, slices):
    from flashmhf_amd import mhffn_backward
    from oracle import mhffn_oracle as orc
    print("case", dh, dims, flush=True)
    B, H, S, E, de, Hk = dims
    ins = make_inputs(B, H, S, dh, E, de, Hk, seed=17, dtype=torch.bfloat16)
    got = mhffn_backward(*(t.to(DEV) for t in ins), grad_w_dtype=torch.float32)
    torch.cuda.synchronize()
    for name, a, r in zip(("dQ", "dK", "dU", "dV", "dR"), got, orc.mhffn_backward(*ins, compute_dtype=torch.float64)):
        assert_bf16_parity(name, a.float().cpu(), r, (dh, dims))
