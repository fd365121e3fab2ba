"""Head prologue at the lines of its rules: forward rows moved whole from 1,024 tiles of 32 tokens on, backward rows from eight waves on with one to three
tiles per wave (workgroups counted heads first) and with more (head by head).  Q, R and dx of a token depend on its own row alone: they agree
bit for bit with calls of few tokens, which move pieces; heads that are no multiple of eight, several batches, last tiles of 1 and 31 rows."""
import pytest
import torch

from .test_gpu_head_gate_rows import _inputs, test_backward as backward_against_pieces

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,H,dh,E,norm", [(1, 4065, 8, 128, 11, True), (3, 1985, 6, 96, 8, True), (2, 4127, 4, 64, 31, True),
                                             (1, 4064, 8, 128, 11, True), (1, 4095, 8, 128, 16, False)])
def test_forward(B, S, H, dh, E, norm):
    from flashmhf_amd.head_gate import head_norm_gate
    print(f"case B={B} S={S} H={H} dh={dh} E={E} norm={norm}", flush=True)
    x, wn, router, _ = _inputs(B, S, H, dh, E, norm)
    Q, R = head_norm_gate(x, wn, router, 1e-6)
    for b in range(B):
        for t in (0, 512, S - 500):
            q, r = head_norm_gate(x[b:b + 1, t:t + 500].contiguous(), wn, router, 1e-6)
            assert torch.equal(Q[b, :, t:t + 500], q[0]) and torch.equal(R[b, :, t:t + 500], r[0])


# one tile per wave: 1,024 tiles, 1,071; two: 2,064 (a second round of workgroups otherwise); three: 6,144; five: 8,256
@pytest.mark.parametrize("B,S,H,dh,E,norm", [(1, 4065, 8, 128, 22, True), (3, 3777, 3, 96, 8, True), (2, 4100, 8, 96, 16, True), (1, 4095, 8, 64, 32, False),
                                             (1, 24570, 8, 64, 5, True), (4, 5473, 12, 128, 11, True)])
def test_backward(B, S, H, dh, E, norm):
    backward_against_pieces(B, S, H, dh, E, norm, True)
