"""Head prologue of the MH-FFN block as one HIP pass each way: per-head RMSNorm of the projected heads
(models/flashmhf/modeling_mhffnmoe.py:97-135, applied at :371-372) and the expert gate
``R = sigmoid(Q router) / max(sum_e, 1e-20)`` (:384-386).

    Q, R = head_norm_gate(x4, norm_weight, router, eps)      # x4 [B,S,H,d_h] bf16 contiguous

``Q`` is the [B,H,S,d_h] *view* of a [B,S,H,d_h] buffer -- the token-major layout the fused operator reads in place --
and ``R`` is [B,H,S,E] float32.  With ``norm_weight=None`` no normalisation happens and Q is a view of ``x4`` itself.
The backward takes dQ (either layout) and dR and returns dx4, d_norm_weight and d_router, recomputing the forward from
``x4``: nothing but the inputs is saved.  bfloat16 only, d_h in {64, 96, 128}, E <= 64; no CPU path.
"""
from . import _capi


def head_norm_gate(x4, norm_weight, router, eps=1e-6):
    return _capi.native().gate(x4, norm_weight, router, float(eps))


class HeadNormGateFunction:
    """The autograd node of ``head_norm_gate`` under the name and call of a torch.autograd.Function."""
    apply = staticmethod(head_norm_gate)
