"""What the performance of this framework is measured on: the calls that a user's program makes, from one decoded token to a
full training batch of the largest layer.

Layer families (the sizes of the configurations, tests and benchmark of this repository; ``head_dim`` etc. per head):

    128M   8 heads of  96,  8 experts of 256 rows          (hidden  768)
    370M   8 heads of 128, 11 experts of 352 rows          (hidden 1024)
    1.3B  16 heads of 128, 22 experts of 352 rows          (hidden 2048)

A case names the entry point it goes through (``kind``, ``entry``), whether it is inference or a training step (``train``:
forward and backward, all gradients), and the extents.  ``kind``:

    op        the fused operator alone: FlashMLPMoE, FlashFFNMoE (float32 weight gradients) or the single-expert FlashMLP
    prologue  head_norm_gate, the per-head RMSNorm and expert gate in front of the operator
    layer     MHFFNLayer: projection, prologue, operator, output projection
    decoder   MHFFNDecoder: attention and MHFFNLayer blocks, loss and the gradients of every parameter
"""
import math

import torch

from flashmhf_amd import FlashFFNMoE, FlashMLP, FlashMLPMoE, MHFFNDecoder, MHFFNLayer
from flashmhf_amd.head_gate import head_norm_gate

DEV = "cuda"
FAMILY = {
    "128M": dict(H=8, Hk=8, dh=96, E=8, de=256),
    "370M": dict(H=8, Hk=8, dh=128, E=11, de=352),
    "1.3B": dict(H=16, Hk=16, dh=128, E=22, de=352),
}


def _op(B, S, train, *, entry="moe", dtype="bf16", token_major=False, **dims):
    return dict(kind="op", entry=entry, train=train, dtype=dtype, token_major=token_major, B=B, S=S, **dims)


def _layer(B, S, train, *, rms=True, **dims):
    return dict(kind="layer", train=train, B=B, S=S, rms=rms, **dims)


def _prologue(B, S, **dims):
    return dict(kind="prologue", train=True, B=B, S=S, **dims)


def _decoder(B, S, blocks, vocab, **dims):
    return dict(kind="decoder", train=True, B=B, S=S, blocks=blocks, vocab=vocab, **dims)


def listed():
    f = FAMILY
    return [
        # Generation, one sequence: the operator on one new token.  The smallest call there is; the weights of every head
        # and expert are read for 8 rows of output.
        dict(_op(1, 1, False, **f["370M"]), name="decode_370m_1"),
        # Generation, a serving batch: the whole block on one new token of each of 16 sequences.
        dict(_layer(16, 1, False, **f["1.3B"]), name="decode_layer_1.3b_16"),
        # Reading one prompt of a length that no tile divides.
        dict(_op(1, 733, False, **f["128M"]), name="prefill_128m_733"),
        # Reading two prompts through the whole block.
        dict(_layer(2, 1500, False, **f["370M"]), name="prefill_layer_370m_2x1500"),
        # Scoring a batch with the 128M layer: the forward benchmark.
        dict(_op(8, 2048, False, **f["128M"]), name="forward_128m_8x2048"),
        # Training the 370M layer on 16,384 tokens: the headline benchmark.
        dict(_op(8, 2048, True, **f["370M"]), name="train_370m_8x2048"),
        # Training the 1.3B layer on 32,768 tokens: the largest call.
        dict(_op(4, 8192, True, token_major=True, **f["1.3B"]), name="train_1.3b_4x8192"),
        # Fine-tuning on a few short ragged sequences, with grouped K/U/V heads and float32 weight gradients.
        dict(_op(2, 300, True, entry="ffn", token_major=True, **dict(f["128M"], Hk=2)), name="finetune_128m_gq_2x300"),
        # The float32 reference configuration (256 tokens of the 128M layer), with gradients.
        dict(_op(2, 128, True, dtype="f32", **f["128M"]), name="train_f32_128m_2x128"),
        # The prologue of the 1.3B layer in training, on the tokens of its benchmark.
        dict(_prologue(4, 8192, **f["1.3B"]), name="prologue_1.3b_4x8192"),
        # One training step of the whole block on a micro-batch.
        dict(_layer(2, 1024, True, **f["370M"]), name="train_layer_370m_2x1024"),
        # One training step of a small decoder: what the block costs among everything else that a model does.
        dict(_decoder(1, 512, 4, 8192, **f["370M"]), name="train_decoder_370m_1x512"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cut(rng, tokens):
    """(B, S) of about `tokens` tokens: one to eight sequences of any length."""
    B = min(tokens, rng.choice([1, 1, 2, 3, 4, 8]))
    return B, max(1, tokens // B)


def draw(rng):
    name = rng.choice(["128M", "370M", "1.3B", "other"])
    if name == "other":
        H = rng.choice([4, 6, 8, 12])
        d = dict(H=H, Hk=rng.choice([H, H, H // 2]), dh=rng.choice([64, 96, 128]), E=rng.randint(2, 16),
                 de=32 * rng.randint(2, 16))
    else:
        d = dict(FAMILY[name])
        if rng.random() < 0.25:
            d["Hk"] = d["H"] // rng.choice([2, 4])
    what = rng.choice(["decode", "decode", "prefill", "prefill", "train", "train", "train", "f32", "prologue", "block",
                       "single", "decoder"])
    rms = rng.random() < 0.75
    if what == "decode":
        B = _log(rng, 1, 64)
        return _layer(B, 1, False, rms=rms, **d) if rng.random() < 0.5 else _op(B, 1, False, **d)
    if what == "prefill":
        B, S = _cut(rng, _log(rng, 16, 16384))
        return _layer(B, S, False, rms=rms, **d) if rng.random() < 0.5 else _op(B, S, False, **d)
    if what == "train":
        B, S = _cut(rng, _log(rng, 128, 16384))
        return _op(B, S, True, entry=rng.choice(["moe", "moe", "ffn"]), token_major=rng.random() < 0.5, **d)
    if what == "f32":
        B, S = _cut(rng, _log(rng, 32, 1024))
        return _op(B, S, rng.random() < 0.7, dtype="f32", **dict(FAMILY["128M"], Hk=rng.choice([8, 4])))
    if what == "prologue":
        B, S = _cut(rng, _log(rng, 512, 32768))
        return _prologue(B, S, **d)
    if what == "block":
        B, S = _cut(rng, _log(rng, 128, 8192))
        return _layer(B, S, True, rms=rms, **d)
    if what == "single":     # the single-expert operator: one feed-forward width per head
        B, S = _cut(rng, _log(rng, 16, 8192))
        d.update(E=1, de=32 * rng.randint(8, 96))
        return _op(B, S, rng.random() < 0.5, entry="mlp", **d)
    B, S = _cut(rng, _log(rng, 128, 2048))
    return _decoder(B, S, rng.randint(1, 4), 32 * rng.randint(64, 256), **FAMILY[rng.choice(["128M", "370M"])])


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _fill(module, g):
    """Parameters with the distributions that the benchmark configurations state, from the generator alone."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if name.endswith("norm.weight"):
                v = 1.0 + 0.1 * torch.randn(p.shape, generator=g, device=DEV)
            elif name.rsplit(".", 1)[-1] in ("K", "U", "V"):
                v = torch.randn(p.shape, generator=g, device=DEV) * p.shape[-1] ** -0.5
            elif "router" in name or "embed" in name:
                v = torch.randn(p.shape, generator=g, device=DEV) * 0.02
            else:
                v = torch.randn(p.shape, generator=g, device=DEV) * p.shape[-1] ** -0.5
            p.copy_(v)


def prepare(case, seed):
    c, g = case, torch.Generator(device=DEV).manual_seed(seed)
    B, S, H, Hk, dh, E, de = (c[k] for k in ("B", "S", "H", "Hk", "dh", "E", "de"))
    st = dict(case=c)
    if c["kind"] == "op":
        dtype = torch.bfloat16 if c["dtype"] == "bf16" else torch.float32
        if c["token_major"]:     # the projection's own memory, seen head by head
            Q, dO = (_normal(g, B, S, H, dh, dtype=dtype).transpose(1, 2) for _ in range(2))
        else:
            Q, dO = (_normal(g, B, H, S, dh, dtype=dtype) for _ in range(2))
        wshape = (Hk, de, dh) if c["entry"] == "mlp" else (Hk, E, de, dh)
        ins = [Q] + [_normal(g, *wshape, std=dh ** -0.5, dtype=dtype) for _ in range(3)]
        if c["entry"] != "mlp":
            R = torch.sigmoid(torch.randn(B, H, S, E, generator=g, device=DEV) * 0.6)
            ins.append(R / R.sum(-1, keepdim=True))
        st["op"] = {"moe": FlashMLPMoE, "ffn": FlashFFNMoE, "mlp": FlashMLP}[c["entry"]]()
        st["ins"] = [t.requires_grad_(c["train"]) for t in ins]
        st["dO"] = dO if c["train"] else None
    elif c["kind"] == "prologue":
        x = _normal(g, B, S, H, dh)
        wn = 1.0 + _normal(g, H, dh, std=0.1, dtype=torch.float32)
        router = _normal(g, H, dh, E, std=0.05)
        st["ins"] = [t.requires_grad_(True) for t in (x, wn, router)]
        st["grads"] = [_normal(g, B, S, H, dh).transpose(1, 2), _normal(g, B, H, S, E, dtype=torch.float32)]
    elif c["kind"] == "layer":
        with torch.device(DEV):
            m = MHFFNLayer(H * dh, H, E, de, Hk, apply_rmsnorm=c["rms"])
        _fill(m, g)
        st["mod"] = m.to(torch.bfloat16).requires_grad_(c["train"])
        st["x"] = _normal(g, B, S, H * dh).requires_grad_(c["train"])
        st["dY"] = _normal(g, B, S, H * dh) if c["train"] else None
    else:
        with torch.device(DEV):
            m = MHFFNDecoder(c["vocab"], H * dh, c["blocks"], H, H, E, de, num_kuv_heads=Hk, apply_rmsnorm=True)
        _fill(m, g)
        st["mod"] = m.to(torch.bfloat16)
        st["ids"] = torch.randint(0, c["vocab"], (B, S), generator=g, device=DEV)
    return st


def run(st):
    c = st["case"]
    if c["kind"] == "op":
        if not c["train"]:
            with torch.no_grad():
                return st["op"](*st["ins"])
        O = st["op"](*st["ins"])
        return [O.detach(), *torch.autograd.grad(O, st["ins"], st["dO"])]
    if c["kind"] == "prologue":
        Q, R = head_norm_gate(*st["ins"], 1e-6)
        return [Q.detach(), R.detach(), *torch.autograd.grad([Q, R], st["ins"], st["grads"])]
    if c["kind"] == "layer":
        if not c["train"]:
            with torch.no_grad():
                return st["mod"](st["x"])
        Y = st["mod"](st["x"])
        return [Y.detach(), *torch.autograd.grad(Y, [st["x"], *st["mod"].parameters()], st["dY"])]
    loss = st["mod"](st["ids"], labels=st["ids"])
    return [loss.detach(), *torch.autograd.grad(loss, list(st["mod"].parameters()))]


def work(case):
    """Bytes: every input read once, every output written once (an inner tensor that two entry points hand on is one of
    neither).  Operations: with F = 2 * tokens * H * E * de * dh for one product, the forward takes 3 F and the backward
    8 F (nothing of the size tokens * E * de may be kept, so its two first products are taken again); an nn.Linear takes one
    product forward and two backward; causal attention half of its square."""
    c = case
    B, S, H, Hk, dh, E, de = (c[k] for k in ("B", "S", "H", "Hk", "dh", "E", "de"))
    T, hid = B * S, H * dh
    F = 2.0 * T * H * E * de * dh
    W, q, r = 3.0 * Hk * E * de * dh, float(T) * hid, 4.0 * T * H * E
    gate = 2.0 * T * hid * E
    if c["kind"] == "op":
        size = 2.0 if c["dtype"] == "bf16" else 4.0
        if c["entry"] == "mlp":
            r = 0.0
        nbytes = size * (2 * q + W) + r
        if c["train"]:
            gw = 4.0 if c["entry"] == "ffn" else size
            nbytes += size * 2 * q + gw * W + r
        return {"bytes": nbytes, "flops": (11 if c["train"] else 3) * F}
    if c["kind"] == "prologue":     # x, Q and R; dQ, dR and dx
        return {"bytes": 2.0 * 4 * q + 2 * r + 2 * (2.0 * hid * E + 4.0 * hid), "flops": 4 * gate}
    lin = 2.0 * T * hid * hid       # one hidden x hidden projection
    params = W + 2.0 * hid * hid + hid * E + (hid if c.get("rms", True) else 0)
    flops = (11 * F + 6 * lin + 4 * gate) if c["train"] else (3 * F + 2 * lin + gate)
    if c["kind"] == "layer":
        return {"bytes": 2.0 * (2 * q + params) * (2 if c["train"] else 1), "flops": flops}
    n, V = c["blocks"], c["vocab"]
    attn = 3 * 4 * lin + 3.5 * (2.0 * B * S * S * hid)
    params = n * (params + 4.0 * hid * hid + 2 * hid) + 2.0 * V * hid + hid
    return {"bytes": 2.0 * 2 * params + 8.0 * T, "flops": n * (flops + attn) + 3 * 2.0 * T * hid * V}


def tolerance(case):
    """float32 in and out: sums in another order.  bfloat16: operands are rounded to 8 bits and so are most outputs; through
    the blocks of a decoder such roundings add up."""
    if case["kind"] == "op" and case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 4e-4}
    return {"rel": 2e-2 if case["kind"] == "decoder" else 1e-2, "max": 0.4 if case["kind"] == "decoder" else 0.2}
