"""The forward of few rows and many blocks: from 32 blocks a part the 32-row tiles take them in a pipeline (csrc/mhffn_fwd.hip).  Numbers of
blocks on both sides of that line and around the pipeline's four waves and five and eight tile sets, experts that end in any of
its phases, rows around a tile and every head width, in one part, against the fp64 oracle; and rows of a larger call, which other
tiles take, bit for bit."""
import pytest
import torch

from oracle import mhffn_oracle as orc
from tests.helpers import assert_bf16_parity, make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("E,de", [(31, 32), (32, 32), (11, 96), (17, 64), (5, 224), (3, 384), (37, 32), (1, 1280), (64, 32)])
def test_blocks_of_the_pipeline(dh, E, de):
    from flashmhf_amd import _capi, mhffn_forward
    S = 33 if E < 17 else 31
    print("case", dh, E, de, S, flush=True)
    plan = _capi.launch_plan(_capi.Dims(1, 2, 1, S, dh, E, de), 0, one_part=True)
    assert (plan.fwd_tile_rows, plan.fwd_parts) == (32, 1)
    ins = make_inputs(1, 2, S, dh, E, de, 1, seed=E, dtype=torch.bfloat16)
    O = mhffn_forward(*(t.to(DEV) for t in ins[:5]), one_part=True)
    torch.cuda.synchronize()
    assert_bf16_parity("O", O.float().cpu(), orc.mhffn_forward(*ins[:5], compute_dtype=torch.float64), (dh, E, de))


@pytest.mark.parametrize("dh", [64, 96, 128])
def test_same_bits_as_larger_tiles(dh):
    from flashmhf_amd import _capi, mhffn_forward
    E, de, few, many = 9, 160, 40, 16000
    plans = [_capi.launch_plan(_capi.Dims(1, 2, 2, S, dh, E, de), 0, one_part=True).fwd_tile_rows for S in (few, many)]
    assert plans[0] == 32 and plans[1] > 32
    Q, K, U, V, R, _ = (t.to(DEV) for t in make_inputs(1, 2, many, dh, E, de, 2, seed=4, dtype=torch.bfloat16))
    large = mhffn_forward(Q, K, U, V, R, one_part=True)
    small = mhffn_forward(Q[:, :, :few].contiguous(), K, U, V, R[:, :, :few].contiguous(), one_part=True)
    torch.cuda.synchronize()
    assert torch.equal(small, large[:, :, :few])
