"""Few rows per head: the forward and the dQ/dR kernel cut the blocks of a head into parts whose fp32 sums a second pass adds
(pick_parts in csrc/mhffn_common.hpp).  Row counts around the 32- and 256-row tiles, tiles that mix batches, q-heads of a
group and ragged ends, parts that begin and end inside an expert, against the fp64 oracle; and MHFFN_ONE_PART, whose
results for a token do not depend on the call's other tokens."""
import pytest
import torch

from oracle import mhffn_oracle as orc
from tests.helpers import assert_bf16_parity, make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    # B, H, S, dh, E, de, Hk, token_major
    (1, 2, 1, 64, 1, 32, 2, False),       # one block: nothing to cut
    (1, 3, 1, 128, 5, 96, 3, True),       # one row, a part per block
    (5, 4, 1, 96, 2, 256, 2, True),       # decoded tokens of five sequences share a tile with the heads of their group
    (1, 2, 255, 128, 3, 224, 2, False),
    (3, 4, 43, 64, 7, 96, 1, False),      # 516 rows of one K/U/V head: tiles across batches and heads
    (1, 8, 1300, 64, 3, 320, 8, True),    # 128-row tiles in two parts
    (1, 1, 129, 128, 2, 64, 1, False),    # a row beyond four 32-row tiles
    (2, 2, 257, 96, 64, 32, 2, False),    # as many experts as one LDS window of gate values holds
]


def _run(case, seed=3):
    B, H, S, dh, E, de, Hk, tm = case
    ins = make_inputs(B, H, S, dh, E, de, Hk, seed=seed, dtype=torch.bfloat16)
    dev = [t.to(DEV) for t in ins]
    if tm:
        dev[0], dev[5] = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (dev[0], dev[5]))
    return ins, dev


@pytest.mark.parametrize("case", CASES)
def test_parts_match_the_oracle(case):
    from flashmhf_amd import _capi, mhffn_backward, mhffn_forward
    print("case", case, flush=True)
    B, H, S, dh, E, de, Hk, _ = case
    assert E * de < 15 * 32 or _capi.lib().mhffn_fwd_workspace_bytes(_capi.Dims(B, H, Hk, S, dh, E, de), 0) > 0
    ins, dev = _run(case)
    O = mhffn_forward(*dev[:5])
    g = mhffn_backward(*dev, grad_w_dtype=torch.float32)
    torch.cuda.synchronize()
    ref = (orc.mhffn_forward(*ins[:5], compute_dtype=torch.float64), *orc.mhffn_backward(*ins, compute_dtype=torch.float64))
    for name, got, r in zip(("O", "dQ", "dK", "dU", "dV", "dR"), (O, *g), ref):
        assert_bf16_parity(name, got.float().cpu(), r, case)


@pytest.mark.parametrize("case", [
    (2, 4, 300, 128, 5, 96, 2, False),        # tiles of 32 rows, four blocks a trip, for all and for few
    (2, 16, 2000, 128, 5, 96, 16, False),     # 256-row tiles against 32-row ones
    (2, 16, 2000, 96, 3, 32, 16, True),       # ... three blocks: a trip that is not full
    (2, 16, 1999, 64, 9, 32, 8, True),        # ... a ragged last tile of two q-heads; a trip of one block
    (1, 8, 1500, 128, 3, 256, 8, False),
])
def test_one_part_does_not_depend_on_the_other_tokens(case):
    from flashmhf_amd import mhffn_backward, mhffn_forward
    _, (Q, K, U, V, R, dO) = _run(case)
    O, g = mhffn_forward(Q, K, U, V, R, one_part=True), mhffn_backward(Q, K, U, V, R, dO, one_part=True)
    few = slice(37, 40)
    q, r, d = (t[-1:, :, few].contiguous() for t in (Q, R, dO))
    o, h = mhffn_forward(q, K, U, V, r, one_part=True), mhffn_backward(q, K, U, V, r, d, one_part=True)
    for a, b in ((o, O), (h[0], g[0]), (h[4], g[4])):
        assert torch.equal(a, b[-1:, :, few])


@pytest.mark.parametrize("entry", ["moe", "ffn", "mlp", "moe function", "ffn function"])
def test_every_operator_offers_one_part(entry):
    from flashmhf_amd import FlashFFNMoE, FlashMLP, FlashMLPMoE
    from flashmhf_amd.flash_ffn_moe_torch import FlashFFNMoEFunction
    from flashmhf_amd.flash_mlp_moe import FlashMLPFunction
    _, (Q, K, U, V, R, dO) = _run((1, 8, 1500, 128, 1 if entry == "mlp" else 11, 352, 8, False))
    op = {"moe": FlashMLPMoE(one_part=True), "ffn": FlashFFNMoE(one_part=True), "mlp": FlashMLP(one_part=True),
          "moe function": lambda *a: FlashMLPFunction.apply(*a, True), "ffn function": lambda *a: FlashFFNMoEFunction.apply(*a, True)}[entry]
    if entry == "mlp":
        K, U, V = (w[:, 0].contiguous() for w in (K, U, V))

    def run(rows):
        leaves = [t[:, :, rows].contiguous().requires_grad_() for t in ([Q] if entry == "mlp" else [Q, R])]
        o = op(leaves[0], K, U, V, *leaves[1:])
        return [o, *torch.autograd.grad(o, leaves, dO[:, :, rows].contiguous())]

    few = slice(37, 40)
    for a, b in zip(run(few), run(slice(None))):
        assert torch.equal(a, b[:, :, few])


@pytest.mark.parametrize("case", [
    # B, H, S, dh, E, de, Hk, token_major: rows around the 128-row tile, weight rows around the 32-row block, every tile width
    (1, 2, 1, 8, 1, 1, 2, False), (1, 2, 127, 32, 2, 31, 1, True), (1, 1, 129, 72, 3, 33, 1, False),
    (2, 2, 64, 128, 5, 65, 2, True), (1, 4, 385, 96, 2, 64, 2, True),
])
def test_float32_parts_and_slices_match_the_oracle(case):
    from flashmhf_amd import mhffn_backward, mhffn_forward
    print("case", case, flush=True)
    B, H, S, dh, E, de, Hk, tm = case
    ins = make_inputs(B, H, S, dh, E, de, Hk, seed=9)
    dev = [t.to(DEV) for t in ins]
    if tm:
        dev[0], dev[5] = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (dev[0], dev[5]))
    got = (mhffn_forward(*dev[:5]), *mhffn_backward(*dev, grad_w_dtype=torch.float32))
    torch.cuda.synchronize()
    ref = (orc.mhffn_forward(*ins[:5], compute_dtype=torch.float64), *orc.mhffn_backward(*ins, compute_dtype=torch.float64))
    for name, a, r in zip(("O", "dQ", "dK", "dU", "dV", "dR"), got, ref):
        err = (a.double().cpu() - r).abs().max().item()
        assert err <= 1e-5 * max(1.0, r.abs().max().item()), (name, case, err)
