"""Drop-in for the reference's ``kernels/triton/flash_mlp_moe.py`` operator boundary
(``FlashMLPFunction`` :739-868, ``FlashMLPMoE`` :871-903), backed by hand-written gfx950 HIP kernels.

    from flashmhf_amd.flash_mlp_moe import FlashMLPMoE
    O = FlashMLPMoE()(Q, K, U, V, R)      # Q [B,H,S,d_h] bf16; K,U,V [Hkuv,E,d_e,d_h] bf16; R [B,H,S,E] fp32

Same call signature, tensor contract, saved tensors (Q, K, U, V, R only -- no activations) and exception types.
Differences, all widening: d_e may be any multiple of 32 (the reference needs 64, :758), the sequence length is
free, R's gradient is exact fp32 instead of bf16-rounded (:542), and all-float32 tensors are accepted (slow exact path).

Q may also be the transposed view of a contiguous [B,S,H,d_h] tensor -- what ``w_self(x).view(B,S,H,d_h).transpose(1,2)``
is before the caller's ``.contiguous()`` (models/flashmhf/modeling_mhffnmoe.py:362,374).  The kernels then read it in place
and O (and dQ) come back in the same token-major layout, so ``O.transpose(1,2).contiguous().view(B,S,hid)`` (:408) copies
nothing.
"""
import torch

from . import _capi


def mhffn_forward(Q, K, U, V, R, one_part=False):
    """Launches the fused forward on the current stream and returns O (same shape and dtype as Q).
    ``one_part``: sum over the experts in one fixed order whatever the number of tokens (MHFFN_ONE_PART in include/mhffn.h)."""
    return _capi.native().op_forward(Q, K, U, V, R, one_part)


def mhffn_backward(Q, K, U, V, R, dO, grad_w_dtype=torch.bfloat16, one_part=False):
    """Launches the fused backward; returns (dQ, dK, dU, dV, dR).  dQ has Q's dtype, dR is fp32,
    dK/dU/dV have ``grad_w_dtype`` (bf16 as flash_mlp_moe.py:808-810, or fp32 as flash_ffn_moe_torch.py:18-20)."""
    assert dO.shape == Q.shape, "grad_output shape should be the same as Q"
    if grad_w_dtype not in (torch.bfloat16, torch.float32):
        _capi.raise_for_code(_capi.ERR_DTYPE, "mhffn_bwd")
    return tuple(_capi.native().op_backward(Q, K, U, V, R, dO, grad_w_dtype == torch.float32, one_part))


class FlashMLPFunction(torch.autograd.Function):
    """forward(ctx, Q, K, U, V, R) -> O ; backward(ctx, dO) -> (dQ, dK, dU, dV, dR).
    Mirrors kernels/triton/flash_mlp_moe.py:739-868.  (The modules record the same node natively, with a tenth of the host
    time, where ``_capi.native_nodes()`` allows it; this class is for the other cases and for callers that use the
    reference's ``FlashMLPFunction.apply``.)"""

    @staticmethod
    def forward(ctx, Q, K, U, V, R, one_part=False):
        O = _capi.traced(mhffn_forward(Q, K, U, V, R, one_part))
        ctx.save_for_backward(Q, K, U, V, R)
        ctx.one_part = one_part
        return O

    @staticmethod
    def backward(ctx, grad_output):
        Q, K, U, V, R = ctx.saved_tensors
        assert grad_output.shape == Q.shape, "grad_output shape should be the same as Q"
        return (*mhffn_backward(Q, K, U, V, R, grad_output, grad_w_dtype=K.dtype, one_part=ctx.one_part), None)


class FlashMLPMoE(torch.nn.Module):
    """Stateless module, ``forward(Q, K, U, V, R) -> O``.  Mirrors kernels/triton/flash_mlp_moe.py:871-903.
    ``one_part``: see ``mhffn_forward``; O, dQ and dR of a token then do not depend, to the last bit, on the other tokens of the
    call.  Without it a call of few rows (below 16,384 per K/U/V head: tokens times the q-heads that share it) adds the sums of several workgroups, in a number and
    so in an order that goes with the number of tokens: faster, and equal up to float32 rounding."""

    one_part = False        # (of modules saved before there was a choice)

    def __init__(self, one_part=False):
        super().__init__()
        self.one_part = one_part

    def forward(self, Q, K, U, V, R):
        if not _capi.native_nodes():
            return FlashMLPFunction.apply(Q, K, U, V, R, self.one_part)
        return _capi.native().op(Q, K, U, V, R, self.one_part)
