"""The float32 kernels, whose products run on the bfloat16 matrix instructions with every operand taken apart into three bfloat16
values, at the edges of their tiles, teams and planes; and values that the taking apart could spoil."""
import math

import pytest
import torch

from oracle import mhffn_oracle as orc
from tests.helpers import make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (B, H, S, d_h, E, d_e, Hk): rows around 1, 32, 128 and 256 per head; one, two and an odd number of blocks (a team of the forward
# has none in the last turn); experts that end inside a block; every column tile, full and not; one part and several
CASES = [(1, 1, 1, 96, 1, 32, 1), (1, 1, 31, 8, 1, 8, 1), (1, 2, 33, 24, 1, 64, 2), (1, 2, 127, 32, 3, 33, 2), (1, 2, 129, 40, 3, 32, 1),
         (2, 1, 128, 64, 2, 95, 1), (1, 4, 257, 72, 5, 40, 2), (1, 1, 65, 96, 7, 31, 1), (3, 2, 43, 88, 2, 97, 2), (1, 1, 200, 128, 3, 70, 1),
         (1, 8, 300, 96, 8, 256, 8)]


def _run(Q, K, U, V, R, dO):
    from flashmhf_amd import mhffn_backward, mhffn_forward
    ins = [t.to(DEV) for t in (Q, K, U, V, R)]
    out = (mhffn_forward(*ins), *mhffn_backward(*ins, dO.to(DEV), grad_w_dtype=torch.float32))
    torch.cuda.synchronize()
    return [t.cpu() for t in out]


@pytest.mark.parametrize("case", CASES)
def test_sums_are_float32_sums(case):
    """Every output's longest sum takes at most `steps` roundings of 2^-24 of its size (six matrix instructions per sixteen terms,
    first over d_h, then over the rows of the experts or the tokens), and the sigmoid and the gate some more; roundings of either
    sign add up as their root."""
    B, H, S, dh, E, de, Hk = case
    print(f"case {case}", flush=True)
    Q, K, U, V, R, dO = make_inputs(B, H, S, dh, E, de, Hk, seed=S + dh, dtype=torch.float32)
    ref = (orc.mhffn_forward(Q, K, U, V, R, compute_dtype=torch.float64), *orc.mhffn_backward(Q, K, U, V, R, dO, compute_dtype=torch.float64))
    terms = dh + max(E * (de + 31), H // Hk * B * S + 31)
    bound = 2.0 ** -24 * (math.sqrt(6 * terms / 16) + 8)
    for name, got, want in zip(("O", "dQ", "dK", "dU", "dV", "dR"), _run(Q, K, U, V, R, dO), ref):
        err = ((got.double() - want.double()).norm() / want.double().norm()).item()
        print(name, err, bound, flush=True)
        assert err <= bound, (name, err, bound)


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("dh", [64, 96, 128])
def test_a_token_without_numbers_stays_alone(dh, value):
    ins = make_inputs(1, 2, 70, dh, 2, 64, 2, seed=3, dtype=torch.float32)
    clean = _run(*ins)
    ins[0][0, 1, 37, 5] = value
    O, dQ, _, _, _, dR = _run(*ins)
    for got, want in ((O, clean[0]), (dQ, clean[1]), (dR, clean[5])):
        assert not torch.isfinite(got[0, 1, 37]).any()
        got[0, 1, 37] = want[0, 1, 37]
        assert torch.equal(got, want)


@pytest.mark.parametrize("dh", [64, 96, 128])
def test_the_largest_numbers_do_not_overflow_when_taken_apart(dh):
    """The largest float32 rounds to a bfloat16 infinity; its planes must not."""
    Q, K, U, V, R, dO = make_inputs(1, 1, 40, dh, 2, 64, 1, seed=4, dtype=torch.float32)
    Q[0, 0, 11, 3] = torch.finfo(torch.float32).max
    K[..., 3] = 2.0 ** -126
    U[..., 3] = 0
    dO[0, 0, 11] *= 2.0 ** -14      # (or dK, dU, the sums of dM and dN times this number, are beyond float32 themselves)
    ref = (orc.mhffn_forward(Q, K, U, V, R, compute_dtype=torch.float64), *orc.mhffn_backward(Q, K, U, V, R, dO, compute_dtype=torch.float64))
    for name, got, want in zip(("O", "dQ", "dK", "dU", "dV", "dR"), _run(Q, K, U, V, R, dO), ref):
        assert torch.isfinite(got).all(), name
        got, want = (t.double().flatten(0, -2) for t in (got, want))      # (column 3 of dK, dU is 2^127 times as large as the others)
        scale = want.abs().amax(0)
        assert ((got - want).abs().amax(0) <= 1e-5 * scale.clamp(min=1e-3)).all(), name
