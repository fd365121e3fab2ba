"""Which kernel a call runs (mhffn_launch_plan), and one case per kernel: the forward's tiles of 256, 128 and 32 rows and those of
dQ/dR of 256 and 32, each in one part and in several, dK/dU/dV in one token slice and in several, for every head width.  The
plan is asserted without a GPU, so that a case whose kernel is no longer picked for it fails instead of testing another one."""
import ctypes

import pytest
import torch

from flashmhf_amd import _capi
from tests.helpers import assert_bf16_parity, make_inputs

DEV = "cuda:0"

# (B, H, S, E, de, Hk): rows of the forward's tile, several parts, rows of dQ/dR's tile, several parts, several token slices
KERNELS = {
    dh: [((1, 1, 129, 1, 32, 1), (128, False, 256, False, False)),
         ((1, 1, 129, 3, 64, 1), (128, True, 256, True, False)),
         ((1, 1, 129, 3, 32, 1), (32, False, 32, False, False)),
         ((1, 1, 300, 9, 256, 1), (32, True, 32, True, False)),
         ((2, 1, 255, 7, 96, 1), (32, True, 32, True, True)),
         ((2, 4, 4097, 1, 32, 2), (256, False, 256, False, True)),
         ((1, 64, 129, 9, 96 if dh == 64 else 256, 64), (256, True, 256, True, False))]
    for dh in (64, 96, 128)
}
CASES = [(dh, dims, want) for dh, cases in KERNELS.items() for dims, want in cases]


def _dims(dh, dims):
    B, H, S, E, de, Hk = dims
    return _capi.Dims(B, H, Hk, S, dh, E, de)


def _plan(d, dtype=_capi.DTYPE_BF16, one_part=False):
    p = _capi.launch_plan(d, dtype, one_part)
    return p.fwd_tile_rows, p.fwd_parts > 1, p.dqdr_tile_rows, p.dqdr_parts > 1, p.dkdudv_slices > 1


@pytest.mark.parametrize("dh,dims,want", CASES)
def test_the_case_runs_the_kernels_it_is_for(dh, dims, want):
    assert _plan(_dims(dh, dims)) == want


def test_the_cases_cover_every_kernel():
    for cases in KERNELS.values():
        plans = [want for _, want in cases]
        assert {p[:2] for p in plans} == {(r, s) for r in (256, 128, 32) for s in (False, True)}
        assert {p[2:4] for p in plans} == {(r, s) for r in (256, 32) for s in (False, True)}
        assert {p[4] for p in plans} == {False, True}


def test_one_part_cases_compare_two_kernels():
    """The cases of test_gpu_parts.test_one_part_does_not_depend_on_the_other_tokens: tile heights of the large call and of the
    small one."""
    from tests.test_gpu_parts import test_one_part_does_not_depend_on_the_other_tokens as t
    cases = [m for m in t.pytestmark if m.name == "parametrize"][0].args[1]
    want = [(32, 32), (256, 256), (256, 256), (256, 256), (128, 32)]
    for (B, H, S, dh, E, de, Hk, _), (fwd, dq) in zip(cases, want, strict=True):
        assert _plan(_capi.Dims(B, H, Hk, S, dh, E, de), one_part=True)[:4] == (fwd, False, dq, False)
        assert _plan(_capi.Dims(1, H, Hk, 3, dh, E, de), one_part=True)[:4] == (32, False, 32, False)


def test_less_workspace_and_one_part_mean_fewer_parts():
    L, p = _capi.lib(), _capi.Plan()
    d = _capi.Dims(1, 8, 8, 512, 128, 11, 352)
    fwd, bwd = (f(d, 0) for f in (L.mhffn_fwd_workspace_bytes, L.mhffn_bwd_workspace_bytes))
    seen = []
    for f in (0, fwd // 2, fwd, 2 * fwd):
        assert L.mhffn_launch_plan(d, 0, f, bwd * f // fwd, 0, p) == 0
        seen.append((p.fwd_parts, p.dqdr_parts))
        assert p.fwd_parts * 4 * 512 * 8 * 128 <= f or p.fwd_parts == 1
        assert L.mhffn_launch_plan(d, 0, f, bwd * f // fwd, _capi.ONE_PART, p) == 0 and p.fwd_parts == p.dqdr_parts == 1
    assert seen[0] == (1, 1) and seen[2] == seen[3] and min(seen[2]) > 1 and seen == sorted(seen)
    sliced = _capi.Dims(2, 8, 2, 300, 96, 8, 256)
    assert L.mhffn_launch_plan(sliced, 0, 0, 0, 0, p) == _capi.ERR_WORKSPACE
    assert L.mhffn_launch_plan(d, 0, 0, 0, 512, p) == _capi.ERR_SHAPE
    assert L.mhffn_launch_plan(d, 7, 0, 0, 0, p) == _capi.ERR_DTYPE
    assert L.mhffn_launch_plan(d, 0, 0, 0, 0, ctypes.POINTER(_capi.Plan)()) == _capi.ERR_NULL_POINTER
    many = _plan(_capi.Dims(1, 8, 8, 33, 128, 65, 32))      # more experts than one LDS window holds: one part, no 32-row tiles
    assert many[:4] == (128, False, 256, False)
    f32 = _capi.launch_plan(_capi.Dims(2, 8, 8, 128, 96, 8, 256), _capi.DTYPE_F32)
    assert f32.fwd_tile_rows == f32.dqdr_tile_rows == 128 and f32.fwd_parts > 1


@pytest.mark.gpu
@pytest.mark.parametrize("dh,dims,want", CASES)
def test_each_kernel_matches_the_oracle(dh, dims, want):
    from flashmhf_amd import mhffn_backward, mhffn_forward
    from oracle import mhffn_oracle as orc
    print("case", dh, dims, flush=True)
    B, H, S, E, de, Hk = dims
    ins = make_inputs(B, H, S, dh, E, de, Hk, seed=5, dtype=torch.bfloat16)
    dev = [t.to(DEV) for t in ins]
    got = (mhffn_forward(*dev[:5]), *mhffn_backward(*dev, grad_w_dtype=torch.float32))
    torch.cuda.synchronize()
    ref = (orc.mhffn_forward(*ins[:5], compute_dtype=torch.float64), *orc.mhffn_backward(*ins, compute_dtype=torch.float64))
    for name, a, r in zip(("O", "dQ", "dK", "dU", "dV", "dR"), got, ref):
        assert_bf16_parity(name, a.float().cpu(), r, (dh, dims))


# (form, in order, M, N, K): both sides of every line of the rule that chooses between the framework's products and the library's
@pytest.mark.parametrize("product,here", [
    (("TN", 0, 1024, 1024, 1), True), (("TN", 1, 1024, 1024, 1 << 20), True), (("TN", 0, 2048, 2056, 300), False), (("TN", 0, 12, 64, 64), False),
    (("NN", 0, 16, 512, 376), True), (("NN", 0, 16, 512, 384), False), (("NN", 0, 17, 512, 1024), True), (("NN", 0, 63, 512, 1032), False),
    (("NN", 0, 64, 512, 1032), True), (("NN", 0, 64, 512, 8192), True),
    (("NT", 0, 2048, 2048, 2048), True), (("NT", 0, 2048, 2048, 2056), False), (("NT", 0, 64, 4096, 4096), True), (("NT", 1, 64, 4096, 4096), False),
    (("NT", 0, 160, 3072, 3072), False), (("NT", 0, 2049, 2048, 64), False), (("NT", 1, 1, 64, 64), True), (("NT", 0, 1, 64, 12), False)])
def test_whose_products_are_faster(product, here):
    form = {"NT": _capi.PRODUCT_NT, "NN": _capi.PRODUCT_NN, "TN": _capi.PRODUCT_TN}[product[0]]
    assert bool(_capi.lib().mhffn_product_faster(form, *product[1:])) is here


# (B, H, S, E, workgroups): two of four waves share a compute unit, one of eight does, and one of four with more than 32 experts
@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("B,H,S,E,workgroups", [(3, 8, 1300, 11, 264), (3, 16, 650, 22, 288), (8, 12, 270, 8, 288), (16, 12, 150, 32, 384), (1, 6, 5392, 11, 258),
                                                (1, 8, 4064, 11, 256), (1, 8, 12288, 11, 192), (1, 8, 4500, 40, 144)])
def test_prologue_backward_has_no_second_round_and_no_idle_half(dh, B, H, S, E, workgroups):
    need = _capi.lib().mhffn_gate_bwd_workspace_bytes(_capi.Dims(B, H, H, S, dh, E, 32))
    assert need == workgroups * (dh * E + dh) * 4      # (a set of partial sums per workgroup)


# (B, H, S, d_h, E, whole rows forward, backward): both sides of 1,024 tiles of 32 tokens, and of the experts that keep to pieces
@pytest.mark.parametrize("B,H,S,dh,E,fwd,bwd", [(1, 8, 4065, 128, 11, True, True), (1, 8, 4064, 128, 11, False, False), (3, 6, 1985, 96, 8, True, True), (2, 4, 4127, 64, 31, True, True),
                                                (1, 8, 4095, 128, 16, True, True), (1, 8, 4095, 64, 32, False, True), (1, 16, 3041, 96, 16, False, True), (1, 16, 3041, 96, 40, False, False),
                                                (3, 3, 3777, 96, 8, True, True), (5, 4, 3300, 64, 8, True, True), (1, 8, 500, 128, 11, False, False), (4, 16, 8192, 128, 22, True, True)])
def test_prologue_moves_whole_rows_of_many_tokens(B, H, S, dh, E, fwd, bwd):
    forms = _capi.launch_forms(_capi.Dims(B, H, H, S, dh, E, 32), _capi.DTYPE_BF16)
    assert bool(forms & _capi.FORM_GATE_FWD_WHOLE_ROWS) is fwd and bool(forms & _capi.FORM_GATE_BWD_WHOLE_ROWS) is bwd


def test_forms_are_refused_as_plans_are():
    L, sliced = _capi.lib(), _capi.Dims(2, 8, 2, 300, 96, 8, 256)
    assert L.mhffn_launch_forms(sliced, 0, 0, 0, 0) == _capi.ERR_WORKSPACE
    assert L.mhffn_launch_forms(sliced, 0, 0, 1 << 30, 512) == _capi.ERR_SHAPE and L.mhffn_launch_forms(sliced, 7, 0, 0, 0) == _capi.ERR_DTYPE
    assert L.mhffn_launch_forms(ctypes.POINTER(_capi.Dims)(), 0, 0, 0, 0) == _capi.ERR_NULL_POINTER
    assert _capi.launch_forms(_capi.Dims(2, 8, 8, 128, 96, 8, 256), _capi.DTYPE_F32) == 0


# (y = x w^T of M x K, one launch for both gradients): both sides of the lines of that rule where dw alone is the library's
@pytest.mark.parametrize("M,N,K,here", [(512, 8192, 1024, True), (2048, 8192, 1024, True), (3000, 8192, 1024, True), (4096, 8192, 1024, False),
                                        (4096, 8192, 768, True), (4096, 16384, 512, True), (4104, 16384, 512, False), (2048, 3072, 2048, False),
                                        (1500, 3072, 2048, True), (512, 8200, 1024, False), (2048, 2048, 2048, True), (8192, 512, 512, True)])
def test_whose_pairs_are_faster(M, N, K, here):
    assert bool(_capi.lib().mhffn_product_pair_faster(0, M, N, K)) is here


# (B, H, S, d_h, E, d_e, Hk, together): parts of dQ, dR and slices of dK, dU, dV of at most 160 MiB lie one behind the other
@pytest.mark.parametrize("B,H,S,dh,E,de,Hk,together", [(2, 8, 300, 96, 8, 256, 2, True), (8, 8, 512, 128, 11, 352, 4, True), (3, 12, 2500, 64, 12, 256, 6, True), (1, 12, 3000, 128, 9, 384, 6, True),
                                                       (4, 12, 1902, 128, 9, 384, 6, False), (2, 12, 2750, 128, 9, 384, 6, False)])
def test_backward_workspace_holds_both_sums_where_one_launch_adds_them(B, H, S, dh, E, de, Hk, together):
    L, d = _capi.lib(), _capi.Dims(B, H, Hk, S, dh, E, de)
    plan = _capi.launch_plan(d, _capi.DTYPE_BF16)
    assert plan.dqdr_parts > 1 and plan.dkdudv_slices > 1
    slices, parts = plan.dkdudv_slices * 3 * Hk * E * de * dh * 4, plan.dqdr_parts * B * H * S * (dh + E) * 4
    assert slices == L.mhffn_bwd_workspace_min_bytes(d, 0)
    assert (slices + parts <= 160 << 20) is together
    assert 0 <= L.mhffn_bwd_workspace_bytes(d, 0) - (slices + parts if together else max(slices, parts)) < 256


@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("H,Hk,S,E,de", [(12, 6, 32, 5, 160), (16, 8, 32, 2, 160), (8, 4, 50, 8, 64), (4, 4, 50, 8, 96), (2, 2, 128, 3, 96), (1, 1, 1, 1, 32)])
def test_dqdr_of_few_rows_has_no_half_empty_large_tiles(dh, H, Hk, S, E, de):
    assert _capi.launch_plan(_capi.Dims(1, H, Hk, S, dh, E, de), _capi.DTYPE_BF16).dqdr_tile_rows == 32
    assert _capi.launch_plan(_capi.Dims(1, H, Hk, S, dh, 65, 32), _capi.DTYPE_BF16).dqdr_tile_rows == 256      # (32-row tiles hold the gates of 64 experts)


# (B, H, Hk, S, d_h, E, d_e, forward, dQ/dR): calls that lower prices of the sums, fitted to others, made slower (tiles of 128 rows in eight parts
# 22.1 us, in six 19.5; of 32 rows in nine 20.4, of 128 in 22 17.4; dQ/dR in three 48.7, in one 45.4) or gave a workspace that they do not need
@pytest.mark.parametrize("B,H,Hk,S,dh,E,de,fwd,dq", [(1, 6, 6, 520, 128, 8, 352, (128, 6), (32, 2)), (47, 16, 8, 1, 128, 22, 352, (128, 22), (32, 10)),
                                                     (36, 16, 8, 1, 128, 22, 352, (128, 22), (32, 10)), (38, 8, 4, 1, 96, 3, 64, (32, 1), (32, 6)),
                                                     (4, 8, 8, 471, 96, 1, 288, (128, 1), (32, 1)), (2, 8, 8, 2568, 128, 9, 320, (256, 1), (256, 1)),
                                                     (4, 8, 8, 2686, 128, 9, 224, (128, 1), (256, 1)), (2, 8, 8, 501, 128, 11, 352, (128, 4), (32, 1))])
def test_parts_only_where_they_pay(B, H, Hk, S, dh, E, de, fwd, dq):
    d = _capi.Dims(B, H, Hk, S, dh, E, de)
    p = _capi.launch_plan(d, _capi.DTYPE_BF16)
    assert (p.fwd_tile_rows, p.fwd_parts) == fwd and (p.dqdr_tile_rows, p.dqdr_parts) == dq
    L = _capi.lib()
    assert L.mhffn_fwd_workspace_bytes(d, 0) == (fwd[1] * B * H * S * dh * 4 if fwd[1] > 1 else 0)
    if dq[1] == 1:
        assert L.mhffn_bwd_workspace_bytes(d, 0) == L.mhffn_bwd_workspace_min_bytes(d, 0)


# (B, H, Hk, S, d_h, E, d_e, rows of a tile) of calls in one part: three rounds of 128-row tiles instead of two of 256, but not four instead of two, nor two instead of one
@pytest.mark.parametrize("B,H,Hk,S,dh,E,de,rows", [(4, 8, 4, 2064, 128, 11, 352, 128), (1, 6, 3, 15528, 64, 11, 320, 128), (8, 8, 8, 1367, 96, 8, 256, 128), (2, 8, 8, 4796, 96, 8, 256, 128),
                                                   (8, 8, 8, 2048, 128, 11, 352, 256), (1, 8, 8, 16384, 96, 8, 256, 256), (4, 16, 16, 8192, 128, 22, 352, 256), (1, 8, 8, 8192, 128, 11, 352, 256)])
def test_forward_in_one_part_has_the_height_with_the_shorter_rounds(B, H, Hk, S, dh, E, de, rows):
    p = _capi.launch_plan(_capi.Dims(B, H, Hk, S, dh, E, de), _capi.DTYPE_BF16)
    assert (p.fwd_tile_rows, p.fwd_parts) == (rows, 1)


# rows of a K/U/V head: up to 32 the forward has no choice but its 32-row tiles, whatever the price of a part of one block
@pytest.mark.parametrize("dh", [64, 96, 128])
@pytest.mark.parametrize("B,H,Hk,E,de", [(2, 8, 4, 8, 256), (1, 4, 2, 14, 96), (32, 6, 6, 3, 384), (16, 4, 2, 5, 128), (1, 1, 1, 1, 32)])
def test_forward_of_few_rows_has_no_large_tiles(dh, B, H, Hk, E, de):
    assert _capi.launch_plan(_capi.Dims(B, H, Hk, 1, dh, E, de), _capi.DTYPE_BF16).fwd_tile_rows == 32
    assert _capi.launch_plan(_capi.Dims(B, H, Hk, 1, dh, 65, 32), _capi.DTYPE_BF16).fwd_tile_rows != 32      # (32-row tiles hold the gates of 64 experts)
