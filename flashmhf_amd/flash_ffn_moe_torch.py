"""Drop-in for the reference's ``kernels/thunderkittens/flash_ffn_moe_torch.py`` (``FlashFFNMoEFunction`` :5-24,
``FlashFFNMoE`` :27-31): same call signature.  That wrapper returns the gradients of the bf16 weights and of Q in float32
(:17-21), and autograd hands each on in its tensor's own dtype: ``FlashFFNMoEFunction`` does as the wrapper does, the
module's native node writes those values without the float32 copies.  The R transpose the ThunderKittens kernel needs
(:9, :23) is not needed here: the HIP kernels read R as [B,H,S,E].
"""
import torch

from . import _capi
from .flash_mlp_moe import mhffn_backward, mhffn_forward


class FlashFFNMoEFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, Q, K, U, V, R, one_part=False):
        O = _capi.traced(mhffn_forward(Q, K, U, V, R, one_part))
        ctx.save_for_backward(Q, K, U, V, R)
        ctx.one_part = one_part
        return O

    @staticmethod
    def backward(ctx, grad_output):
        Q, K, U, V, R = ctx.saved_tensors
        dQ, dK, dU, dV, dR = mhffn_backward(Q, K, U, V, R, grad_output, grad_w_dtype=torch.float32, one_part=ctx.one_part)
        return dQ.float(), dK, dU, dV, dR, None


class FlashFFNMoE(torch.nn.Module):
    """``one_part``: as in ``FlashMLPMoE``."""

    one_part = False        # (of modules saved before there was a choice)

    def __init__(self, one_part=False):
        super().__init__()
        self.one_part = one_part

    def forward(self, Q, K, U, V, R):
        if not _capi.native_nodes():
            return FlashFFNMoEFunction.apply(Q, K, U, V, R, self.one_part)
        return _capi.native().op(Q, K, U, V, R, self.one_part)
