"""mhffn_bwd with any workspace from the smallest it accepts to the one it asks for: the same gradients up to the order of
float32 sums, and not a byte written behind the workspace."""
import pytest
import torch

from tests.helpers import make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _bwd(L, ins, dims, wdtype, ws_bytes, phases=None):
    from flashmhf_amd import _capi
    Q, K, U, V, R, dO = ins
    outs = [torch.full_like(Q, float("nan")), *(torch.full(K.shape, float("nan"), dtype=wdtype, device=DEV) for _ in range(3)),
            torch.full_like(R, float("nan"))]
    ws = torch.full((ws_bytes + 4096,), 165, dtype=torch.uint8, device=DEV)
    rc = L.mhffn_bwd_layout(*(t.data_ptr() for t in (*ins, *outs)), _capi.torch_dtype_code(wdtype), ws.data_ptr() if ws_bytes else None,
                            ws_bytes, dims, _capi.torch_dtype_code(Q.dtype), 0, torch.cuda.current_stream().cuda_stream,
                            _capi.BWD_ALL if phases is None else phases)
    torch.cuda.synchronize()
    assert rc != 0 or (ws[ws_bytes:] == 165).all()
    return rc, outs


@pytest.mark.parametrize("shape,dtype", [
    ((1, 8, 512, 128, 11, 352, 8), torch.bfloat16),      # one token slice: a NULL workspace will do
    ((1, 16, 1, 128, 22, 352, 16), torch.bfloat16),
    ((2, 8, 300, 96, 8, 256, 2), torch.bfloat16),        # token slices
    ((3, 4, 43, 64, 7, 96, 1), torch.bfloat16),
    ((2, 4, 60, 40, 40, 7, 2), torch.float32),
])
def test_backward_runs_with_less_workspace(shape, dtype):
    from flashmhf_amd import _capi
    print("case", shape, dtype, flush=True)
    L = _capi.lib()
    B, H, S, dh, E, de, Hk = shape
    ins = [t.to(DEV) for t in make_inputs(B, H, S, dh, E, de, Hk, seed=1, dtype=dtype)]
    dims, code = _capi.Dims(B, H, Hk, S, dh, E, de), _capi.torch_dtype_code(dtype)
    need, most = L.mhffn_bwd_workspace_min_bytes(dims, code), L.mhffn_bwd_workspace_bytes(dims, code)
    rc, want = _bwd(L, ins, dims, dtype, most)
    assert rc == 0
    for ws_bytes in sorted({need, need + (most - need) // 3 // 16 * 16, most + 1024}):
        rc, got = _bwd(L, ins, dims, dtype, ws_bytes)
        assert rc == 0, (ws_bytes, _capi.strerror(rc))
        for name, a, b in zip(("dQ", "dK", "dU", "dV", "dR"), got, want):
            # the same terms in another order: float32 results move by a few units of 2^-24 of their terms' size, bfloat16
            # ones by one rounding, 2^-8 of the value
            tol = 2 ** -8 if a.dtype == torch.bfloat16 else 1e-5
            err = (a.float() - b.float()).abs().max().item()
            assert err <= tol * b.float().abs().max().item(), (name, ws_bytes, err)
        if ws_bytes == need:
            rc, one = _bwd(L, ins, dims, dtype, need, _capi.BWD_ALL | 256)       # MHFFN_ONE_PART: needs no more either
            assert rc == 0 and all(not t.isnan().any() for t in one)
            if need == 0:
                assert all(torch.equal(a, b) for a, b in zip(one, got))
    if need:
        assert _bwd(L, ins, dims, dtype, need - 16)[0] == _capi.ERR_WORKSPACE


@pytest.mark.parametrize("shape", [(2, 8, 300, 96, 8, 256, 2), (3, 4, 43, 64, 7, 96, 1), (1, 1, 700, 128, 9, 256, 1)])
@pytest.mark.parametrize("weights", [torch.bfloat16, torch.float32])
def test_sums_in_one_launch_have_the_bits_of_two(shape, weights):
    """With room for the parts of dQ, dR behind the token slices of dK, dU, dV one launch adds up both; with less they take turns."""
    from flashmhf_amd import _capi
    print("case", shape, weights, flush=True)
    L = _capi.lib()
    B, H, S, dh, E, de, Hk = shape
    dims, code = _capi.Dims(B, H, Hk, S, dh, E, de), _capi.DTYPE_BF16
    plan = _capi.launch_plan(dims, code)
    assert plan.dqdr_parts > 1 and plan.dkdudv_slices > 1
    ins = [t.to(DEV) for t in make_inputs(B, H, S, dh, E, de, Hk, seed=2, dtype=torch.bfloat16)]
    most = L.mhffn_bwd_workspace_bytes(dims, code)
    results = [_bwd(L, ins, dims, weights, b) for b in (most, most - 256)]
    assert [rc for rc, _ in results] == [0, 0]
    assert all(torch.equal(a, b) for a, b in zip(results[0][1], results[1][1]))
