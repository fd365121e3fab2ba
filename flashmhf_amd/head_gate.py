"""Head prologue of the MH-FFN block as one HIP pass each way: per-head RMSNorm of the projected heads
(models/flashmhf/modeling_mhffnmoe.py:97-135, applied at :371-372) and the expert gate
``R = sigmoid(Q router) / max(sum_e, 1e-20)`` (:384-386).

    Q, R = head_norm_gate(x4, norm_weight, router, eps)      # x4 [B,S,H,d_h] bf16 contiguous

``Q`` is the [B,H,S,d_h] *view* of a [B,S,H,d_h] buffer -- the token-major layout the fused operator reads in place --
and ``R`` is [B,H,S,E] float32.  With ``norm_weight=None`` no normalisation happens and Q is a view of ``x4`` itself.
The backward takes dQ (either layout) and dR and returns dx4, d_norm_weight and d_router, recomputing the forward from
``x4``: nothing but the inputs is saved.  bfloat16 only, d_h in {64, 96, 128}, E <= 64; no CPU path.
"""
import torch

from . import _capi


class HeadNormGateFunction(torch.autograd.Function):
    """The node of ``head_norm_gate`` as a torch.autograd.Function, for where the native one cannot run
    (``_capi.native_nodes``)."""

    @staticmethod
    def forward(ctx, x4, norm_weight, router, eps):
        ctx.save_for_backward(x4, norm_weight, router)
        ctx.eps = float(eps)
        Q, R = _capi.native().gate(x4, norm_weight, router, ctx.eps)
        return _capi.traced(Q), _capi.traced(R)

    @staticmethod
    def backward(ctx, dQ, dR):
        x4, norm_weight, router = ctx.saved_tensors
        return (*_capi.native().gate_backward(x4, norm_weight, router, ctx.eps, dQ, dR), None)


def head_norm_gate(x4, norm_weight, router, eps=1e-6):
    if not _capi.native_nodes():
        return HeadNormGateFunction.apply(x4, norm_weight, router, eps)
    return _capi.native().gate(x4, norm_weight, router, float(eps))
