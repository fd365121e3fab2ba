"""dQ and dR of few rows: the 32-row kernel takes the blocks of a head in a pipeline (csrc/mhffn_bwd.hip).  Numbers of blocks around
the pipeline's four waves and seven tile sets, experts that end in any of its phases, rows around a tile and every head width,
in one part, against the fp64 oracle."""
import pytest
import torch

from oracle import mhffn_oracle as orc
from tests.helpers import assert_bf16_parity, make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("E,de", [(1, 32), (2, 32), (3, 32), (1, 128), (5, 32), (2, 96), (7, 32), (1, 256), (3, 96), (5, 64), (5, 96), (64, 32)])
def test_blocks_of_the_pipeline(dh, E, de):
    from flashmhf_amd import _capi, mhffn_backward
    S = 33 if E < 5 else 31
    print("case", dh, E, de, S, flush=True)
    if E * de > 32:
        assert _capi.launch_plan(_capi.Dims(1, 2, 1, S, dh, E, de), 0, one_part=True).dqdr_tile_rows == 32
    ins = make_inputs(1, 2, S, dh, E, de, 1, seed=E, dtype=torch.bfloat16)
    dQ, _, _, _, dR = mhffn_backward(*(t.to(DEV) for t in ins), grad_w_dtype=torch.float32, one_part=True)
    torch.cuda.synchronize()
    ref = orc.mhffn_backward(*ins, compute_dtype=torch.float64)
    assert_bf16_parity("dQ", dQ.float().cpu(), ref[0], (dh, E, de))
    assert_bf16_parity("dR", dR.float().cpu(), ref[4], (dh, E, de))
