"""dK/dU/dV with two waves for a block of rows, each on half of the slice's tokens (TokenHalves in csrc/mhffn_bwd.hip): numbers of tiles that
do not halve, a block alone in its workgroup, sequences of one row and ragged ends, grouped heads, both layouts, several slices."""
import pytest
import torch

from flashmhf_amd import _capi
from tests.helpers import assert_bf16_parity, make_inputs

DEV = "cuda:0"

# B, H, S, E, de, Hk, token slices of such workgroups
CASES = [
    (1, 2, 192, 1, 96, 2, 1),       # six tiles; three blocks: the last workgroup of a head has one
    (1, 3, 223, 1, 32, 3, 1),       # four tiles and three; a ragged end; one block
    (7, 2, 1, 3, 64, 2, 1),         # tiles of one row
    (3, 4, 40, 2, 96, 2, 1),        # 12 tiles of two heads and three sequences
    (1, 8, 1000, 8, 256, 8, 1),     # the other form would take two slices
    (2, 8, 300, 8, 256, 2, 4),      # 80 tiles in slices of 20
    (3, 4, 170, 3, 96, 4, 2),       # 18 tiles in slices of nine, five of them and four; the last workgroup of a head has one block
    (2, 3, 288, 5, 96, 3, 2),       # whole tiles, 18 in slices of nine; 15 blocks
    (2, 4, 136, 1, 384, 2, 2),      # a ragged end, 20 tiles in slices of ten
    (3, 6, 210, 3, 96, 3, 5),       # 42 tiles in slices of eight and nine, the latter five tiles and four; nine blocks
]


@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("case", CASES)
def test_slices(case, dh):
    B, H, S, E, de, Hk, slices = case
    d = _capi.Dims(B, H, Hk, S, dh, E, de)
    assert _capi.launch_forms(d, _capi.DTYPE_BF16) & _capi.FORM_TOKEN_HALVES
    assert _capi.launch_plan(d, _capi.DTYPE_BF16).dkdudv_slices == slices


# columns that fill the chip, few tiles, and longer steps that cost more than half the partial sums save
@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("B,H,S,E,de,Hk", [(8, 8, 2048, 11, 352, 8), (1, 2, 32, 1, 96, 2), (1, 1, 64, 1, 32, 1), (4, 1, 8, 3, 64, 1), (1, 8, 128, 8, 256, 8)])
def test_the_other_form_runs_elsewhere(B, H, S, E, de, Hk, dh):
    assert not _capi.launch_forms(_capi.Dims(B, H, Hk, S, dh, E, de), _capi.DTYPE_BF16) & _capi.FORM_TOKEN_HALVES


@pytest.mark.gpu
@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("case", CASES)
def test_gradients_match_the_oracle(case, dh):
    from flashmhf_amd import mhffn_backward
    from oracle import mhffn_oracle as orc
    print("case", case, dh, flush=True)
    B, H, S, E, de, Hk, _ = case
    ins = make_inputs(B, H, S, dh, E, de, Hk, seed=11, dtype=torch.bfloat16)
    ref = orc.mhffn_backward(*ins, compute_dtype=torch.float64)
    dev = [t.to(DEV) for t in ins]
    rows = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in (dev[0], dev[5])]       # token-major: the same bits
    got = {w: mhffn_backward(*dev, grad_w_dtype=w) for w in (torch.float32, torch.bfloat16)}
    again = mhffn_backward(rows[0], *dev[1:5], rows[1], grad_w_dtype=torch.float32)
    torch.cuda.synchronize()
    for w, g in got.items():
        for name, a, r in zip(("dQ", "dK", "dU", "dV", "dR"), g, ref):
            assert_bf16_parity(name, a.float().cpu(), r, (case, dh, w))
    for a, b, c in zip(got[torch.float32][1:4], again[1:4], got[torch.bfloat16][1:4]):
        assert torch.equal(a, b) and torch.equal(a.bfloat16(), c)
