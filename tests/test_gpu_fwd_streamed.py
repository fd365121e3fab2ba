"""The forward of few rows with weights larger than the L2 caches together and, from 64 MiB on, read past the caches by the 32-row tiles
(csrc/mhffn_fwd.hip, fwd_reads_past).  Weights just above and just below these sizes, rows around a tile, parts that end in the middle of a trip, grouped heads and every head
width, against the fp64 oracle."""
import pytest
import torch

from oracle import mhffn_oracle as orc
from tests.helpers import assert_bf16_parity, make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
L2 = 8 * 4 << 20


@pytest.mark.parametrize("H,Hkuv,S,dh,E,de,past", [(8, 8, 1, 128, 22, 352, True), (8, 8, 33, 128, 16, 352, True), (8, 8, 32, 128, 11, 480, False),
                                                   (8, 8, 31, 128, 11, 512, True), (16, 8, 2, 128, 17, 352, True), (16, 16, 5, 64, 22, 352, True),
                                                   (16, 16, 33, 64, 17, 320, False), (8, 8, 1, 96, 16, 512, True), (16, 16, 30, 96, 13, 288, True)])
def test_few_rows(H, Hkuv, S, dh, E, de, past):
    from flashmhf_amd import _capi, mhffn_forward
    print("case", H, Hkuv, S, dh, E, de, flush=True)
    plan = _capi.launch_plan(_capi.Dims(1, H, Hkuv, S, dh, E, de), 0)
    assert plan.fwd_tile_rows == 32 and E * de // 32 // plan.fwd_parts < 32
    assert (3 * Hkuv * E * de * dh * 2 > L2) == past
    ins = make_inputs(1, H, S, dh, E, de, Hkuv, seed=E, dtype=torch.bfloat16)
    O = mhffn_forward(*(t.to(DEV) for t in ins[:5]))
    torch.cuda.synchronize()
    assert_bf16_parity("O", O.float().cpu(), orc.mhffn_forward(*ins[:5], compute_dtype=torch.float64), (H, S, dh, E, de))


@pytest.mark.parametrize("H,Hkuv,S,dh,E,de,past", [(16, 16, 1, 128, 22, 352, True), (16, 16, 33, 128, 17, 352, True), (16, 16, 31, 128, 16, 352, True), (32, 16, 2, 128, 15, 384, True),
                                                   (16, 16, 32, 128, 15, 352, False), (32, 32, 5, 64, 16, 352, True), (32, 32, 5, 64, 15, 352, False),
                                                   (16, 16, 30, 96, 22, 352, True), (16, 16, 33, 96, 20, 352, False), (8, 8, 1, 128, 22, 352, False)])
def test_past_the_caches(H, Hkuv, S, dh, E, de, past):
    from flashmhf_amd import _capi
    assert bool(_capi.launch_forms(_capi.Dims(1, H, Hkuv, S, dh, E, de), 0) & _capi.FORM_WEIGHTS_PAST_CACHES) == past == (3 * Hkuv * E * de * dh * 2 > 64 << 20)
    test_few_rows(H, Hkuv, S, dh, E, de, 3 * Hkuv * E * de * dh * 2 > L2)
