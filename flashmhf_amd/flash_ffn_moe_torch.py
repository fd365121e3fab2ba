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
    def forward(ctx, Q, K, U, V, R):
        O = _capi.traced(mhffn_forward(Q, K, U, V, R))
        ctx.save_for_backward(Q, K, U, V, R)
        return O

    @staticmethod
    def backward(ctx, grad_output):
        Q, K, U, V, R = ctx.saved_tensors
        dQ, dK, dU, dV, dR = mhffn_backward(Q, K, U, V, R, grad_output, grad_w_dtype=torch.float32)
        return dQ.float(), dK, dU, dV, dR


class FlashFFNMoE(torch.nn.Module):
    def __init__(self):
        super().__init__()

    def forward(self, Q, K, U, V, R):
        if not _capi.native_nodes():
            return FlashFFNMoEFunction.apply(Q, K, U, V, R)
        return _capi.native().op(Q, K, U, V, R, False)
