"""The float32 operator at the ends of its range: what a float32 evaluation of the same formulas gives there is also what the kernels
give, whatever instructions their products run on."""
import math

import pytest
import torch

from oracle import mhffn_oracle as orc
from tests.helpers import make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ("O", "dQ", "dK", "dU", "dV", "dR")


def _run(Q, K, U, V, R, dO):
    from flashmhf_amd import mhffn_backward, mhffn_forward
    ins = [t.to(DEV) for t in (Q, K, U, V, R)]
    out = (mhffn_forward(*ins), *mhffn_backward(*ins, dO.to(DEV), grad_w_dtype=torch.float32))
    torch.cuda.synchronize()
    return [t.cpu() for t in out]


def _oracle(*ins):
    return (orc.mhffn_forward(*ins[:5], compute_dtype=torch.float64), *orc.mhffn_backward(*ins, compute_dtype=torch.float64))


def _error(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


def _bound(B, H, S, dh, E, de, Hk):
    """Roundings of 2^-24 of the size of the longest sum, of either sign (see test_gpu_f32_split.py)."""
    return 2.0 ** -24 * (math.sqrt(6 * (dh + max(E * (de + 31), H // Hk * B * S + 31)) / 16) + 8)


@pytest.mark.parametrize("value", [-1e2, -1e10, -1e37, torch.finfo(torch.float32).min])
@pytest.mark.parametrize("dh", [64, 96, 128])
def test_silu_goes_to_zero(dh, value):
    """Rows of K that mask their hidden unit (a constant column of Q times a very negative number): SiLU and its derivative are zero."""
    shape = B, H, S, dh, E, de, Hk = 1, 2, 70, dh, 2, 64, 2
    print(f"case d_h={dh} value={value}", flush=True)
    ins = make_inputs(B, H, S, dh, E, de, Hk, seed=9, dtype=torch.float32)
    ins[0][..., 3] = 1.0
    ins[1][:, :, ::5] = 0.0
    ins[1][:, :, ::5, 3] = value
    want = _oracle(*ins)
    for name, got, ref in zip(NAMES, _run(*ins), want):
        assert torch.isfinite(got).all(), name
        assert _error(got, ref) <= _bound(*shape), (name, _error(got, ref))
    got = _run(*ins)
    assert (got[2][:, :, ::5].abs() <= 1e-30).all() and (got[4][:, :, ::5].abs() <= 1e-30).all()      # (masked rows of dK, dV)


@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("dh", [64, 128])
def test_saturated_preactivations(dh, sign):
    """Pre-activations of a few hundred of either sign, zero gates and zero rows."""
    shape = B, H, S, dh, E, de, Hk = 2, 2, 96, dh, 3, 64, 2
    Q, K, U, V, R, dO = make_inputs(B, H, S, dh, E, de, Hk, seed=5, dtype=torch.float32)
    Q, K = Q * 12.0 * sign, K * 4.0
    Q[:, :, 5] = 0
    R[:, :, ::3, 1] = 0.0
    R[:, :, 7] = 0.0
    assert torch.einsum("bhsd,hejd->bhsej", Q, K).abs().max() > 150
    out = _run(Q, K, U, V, R, dO)
    assert torch.equal(out[0][:, :, 7], torch.zeros(B, H, dh))
    # the sigmoid of a pre-activation m is off by |m| times m's own relative rounding: 2^-24 of a few hundred
    for name, got, ref in zip(NAMES, out, _oracle(Q, K, U, V, R, dO)):
        assert torch.isfinite(got).all(), name
        assert _error(got, ref) <= 16 * _bound(*shape), (name, _error(got, ref))


def _same_with_infinities(name, got, want):
    """Infinities and NaN in the same places, and the rest alike."""
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(got), kind(want)), (name, kind, kind(got).sum(), kind(want).sum())
    ok = torch.isfinite(want)
    if ok.any():
        assert _error(got[ok], want[ok].double()) <= 1e-5, name


def _eager(Q, K, U, V, R, dO):
    return (orc.mhffn_forward(Q, K, U, V, R, compute_dtype=torch.float32), *orc.mhffn_backward(Q, K, U, V, R, dO, compute_dtype=torch.float32))


@pytest.mark.parametrize("value", [float("inf"), -float("inf")])
@pytest.mark.parametrize("B,H,S,dh,E,de", [(1, 2, 70, 24, 2, 40), (1, 2, 70, 64, 2, 64), (1, 1, 130, 96, 3, 64), (1, 1, 300, 96, 8, 256), (1, 2, 45, 128, 2, 72)])
def test_an_infinite_weight(B, H, S, dh, E, de, value):
    """One infinite value of V: infinities of the signs that float32 arithmetic gives in O, dQ and dR, and NaN in its rows of dK and dU."""
    print(f"case S={S} d_h={dh} E={E} d_e={de} value={value}", flush=True)
    ins = make_inputs(B, H, S, dh, E, de, H, seed=dh, dtype=torch.float32)
    ins[3][H - 1, E - 1, 37, dh - 2] = value
    for name, got, want in zip(NAMES, _run(*ins), _eager(*ins)):
        _same_with_infinities(name, got, want)
        assert torch.isfinite(got[:, 0]).all() if H > 1 and name in ("O", "dQ", "dR") else not torch.isfinite(got).all() or name == "dV"


@pytest.mark.parametrize("dh", [24, 64, 96, 128])
def test_products_beyond_the_largest_number(dh):
    """SiLU(M) N overflows for two tokens, from finite operands: O has their infinities, and the gradients' rows what float32 gives."""
    Q, K, U, V, R, dO = (t.abs() for t in make_inputs(1, 2, 70, dh, 2, 64, 2, seed=6, dtype=torch.float32))
    Q[0, 1, 5] *= 1e22
    Q[0, 1, 40] *= 1e25
    V[:, :, :, 1] *= -1
    got, want = _run(Q, K, U, V, R, dO), _eager(Q, K, U, V, R, dO)
    assert torch.isposinf(want[0][0, 1, 5, 0]) and torch.isneginf(want[0][0, 1, 5, 1])
    for name, a, b in zip(NAMES, got, want):
        _same_with_infinities(name, a, b)


@pytest.mark.parametrize("dh", [16, 64, 96, 128])
def test_products_are_not_cut_to_one_side(dh):
    """Operands just below 1 + 2^-7, whose product loses most when they are taken apart, times powers of two that add up to a number of
    eight bits in the first product alone; N and V are such numbers, too.  What is left out of a product is at most 2^-24 of it; beside that a
    value of O has seven roundings of at most 2^-24 (M, e^-M and the sigmoid, SiLU, times N, times V), of which the mean over 1,024 values is
    far below half of one."""
    H, S, de = 4, 256, 1
    g = torch.Generator().manual_seed(1)
    eight_bits = lambda *shape: torch.randint(128, 256, shape, generator=g)
    weight, at = eight_bits(1, H, S), 1 + 2.0 ** -7 - 2.0 ** -16
    Q, K, U, V = torch.zeros(1, H, S, dh), torch.zeros(H, 1, de, dh), torch.zeros(H, 1, de, dh), torch.zeros(H, 1, de, dh)
    for c in range(8):
        Q[..., c] = (weight >> c & 1) * 2.0 ** (c - 5) * (at + 2.0 ** -23 * torch.arange(S))
    K[..., :8] = at
    Q[..., 8] = eight_bits(1, H, S) / 128
    U[..., 8] = eight_bits(H, 1, de) / 128
    V[..., 0] = eight_bits(H, 1, de) / 128
    ins = (Q, K, U, V, torch.ones(1, H, S, 1))
    want = orc.mhffn_forward(*ins, compute_dtype=torch.float64)[..., 0]
    got = _run(*ins, torch.ones(1, H, S, dh))[0][..., 0]
    off = ((got.double() - want) / want).mean().item() * 2 ** 24
    print("mean error in 2^-24:", off, flush=True)
    assert abs(off) <= 1.5


# powers of two that Q, K and U, V, R, dO are multiplied by
SMALL = [(0, 0, 0, 0, -114), (0, 0, -114, 0, 0), (0, 0, 0, -114, 0), (-114, 90, 0, 0, 0), (90, -114, 0, 0, 0), (0, 0, 0, -100, -14), (-10, 0, -60, 0, -30)]


@pytest.mark.parametrize("powers", SMALL)
@pytest.mark.parametrize("dh", [24, 64, 96, 128])
def test_small_numbers_keep_their_bits(dh, powers):
    """Operands, and values between the products, a few powers of two above the smallest normal number: results have the relative error
    of ordinary ones wherever they are well above that number themselves."""
    shape = B, H, S, dh, E, de, Hk = 1, 2, 70, dh, 2, 64, 2
    print(f"case d_h={dh} powers={powers}", flush=True)
    Q, K, U, V, R, dO = make_inputs(B, H, S, dh, E, de, Hk, seed=8, dtype=torch.float32)
    q, ku, v, r, do = (2.0 ** p for p in powers)
    ins = (Q * q, K * ku, U * ku, V * v, R * r, dO * do)
    checked = 0
    for name, got, want in zip(NAMES, _run(*ins), _oracle(*ins)):
        if want.abs().max() < 2.0 ** -117:      # (most of it would be denormal: those have fewer bits)
            continue
        checked += 1
        assert _error(got, want) <= _bound(*shape), (name, _error(got, want), want.abs().max())
    assert checked >= 3


# (B, H, S, d_h, E, d_e, Hk, parts of one block): such parts run on the fp32 instructions, and dK, dU, dV of d_h <= 32 with one step a slice
@pytest.mark.parametrize("B,H,S,dh,E,de,Hk,one", [(1, 1, 1, 8, 1, 8, 1, True), (1, 2, 129, 32, 1, 33, 2, True), (1, 8, 63, 96, 8, 256, 4, True), (2, 4, 16, 64, 4, 120, 4, True),
                                                  (1, 1, 65, 128, 2, 32, 1, True), (1, 8, 65, 96, 8, 256, 8, False), (1, 2, 700, 24, 3, 70, 1, True), (1, 1, 66, 16, 1, 32, 1, True)])
def test_parts_of_one_block_and_of_more(B, H, S, dh, E, de, Hk, one):
    from flashmhf_amd import _capi
    print("case", B, H, S, dh, E, de, Hk, flush=True)
    plan = _capi.launch_plan(_capi.Dims(B, H, Hk, S, dh, E, de), _capi.DTYPE_F32)
    assert (plan.fwd_parts == E * ((de + 31) // 32)) is one and (plan.dqdr_parts == plan.fwd_parts or not one)
    ins = make_inputs(B, H, S, dh, E, de, Hk, seed=S, dtype=torch.float32)
    bound = 2.0 ** -24 * (math.sqrt((dh + max(E * (de + 31), H // Hk * B * S + 31)) / 2) + 8)      # (_bound, with one rounding per two terms)
    for name, got, want in zip(NAMES, _run(*ins), _oracle(*ins)):
        assert _error(got, want) <= bound, (name, _error(got, want))
    ins[3][0, 0, 3, dh - 2] = float("inf")      # (of d_h that is no multiple of 32 the first four columns stand in for those beyond it, times zero)
    for name, got, want in zip(NAMES, _run(*ins), _eager(*ins)):
        if name in ("O", "dQ", "dR"):           # (the rows that a tile lacks are others times zero in dK, dU, dV)
            _same_with_infinities(name, got, want)
