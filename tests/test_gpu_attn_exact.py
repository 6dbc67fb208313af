"""Attention calls whose weights are fp32 from the scores to the last product
(fp32 and ragged fp16 operands, bf16 heads of 32, explicit masks, dropout):
their precision, and infinities and NaN in rows that a query does not see."""
from __future__ import annotations

import math

import pytest
import torch

from lzhip import ops

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _heads(t, B, S, n, hd):
    return t.double().cpu().view(B, S, n, hd).transpose(1, 2)


def _call(qkv, do, B, S, H, KV, hd, mask, p=0.0, key=0):
    """(o, lse, dq, dk, dv) through the entry points the layer takes."""
    q2, k2, v2 = qkv[:, : H * hd], qkv[:, H * hd : (H + KV) * hd], qkv[:, (H + KV) * hd :]
    d = torch.zeros_like(qkv)
    grads = d[:, : H * hd], d[:, H * hd : (H + KV) * hd], d[:, (H + KV) * hd :]
    scale = hd**-0.5
    if mask is None and p == 0.0:
        o, lse = ops.attn_fwd_direct(q2, k2, v2, B, S, H, KV, hd, scale)
        ops.attn_bwd_direct(q2, k2, v2, o, do, lse, B, S, H, KV, hd, scale, *grads)
    else:
        o, lse = ops.attn_fwd_general(q2, k2, v2, B, S, H, KV, hd, scale, mask, p, key)
        ops.attn_bwd_general(q2, k2, v2, o, do, lse, B, S, H, KV, hd, scale, *grads, mask, p, key)
    return o, lse, *grads


@pytest.mark.parametrize("masked,hd", [(False, 32), (True, 32), (True, 64), (True, 128)])
def test_bf16_weights_keep_their_fp32_bits(masked, hd):
    """Every output is a difference of nearly equal probabilities: keys come
    in pairs (one bf16 ulp apart in one small column, V of opposite sign) and
    so do queries (dO of opposite sign), so O, dQ, dK and dV are about 1e-4 of
    the weights they are formed from.  Rounding an output to bf16 costs
    2^-9 / sqrt(3) of it (0.11 %), weights good to a few fp32 ulps
    4 * 2^-24 / 1e-4 (0.24 %); weights of 17 bits would cost 2 %."""
    S, n = 64, 32  # keys below n, queries from n on: every query sees every key
    g = torch.Generator().manual_seed(hd + masked)
    q, k, v, do = (torch.zeros(S, hd) for _ in range(4))

    def pairs(rows, small, step):
        x = torch.randn(n // 2, hd, generator=g).to(BF16).float()
        x[:, small] = {32: 0.0625, 64: 0.09375, 128: 0.125}[hd] * (1 - 2 * torch.randint(0, 2, (n // 2,), generator=g))
        x[:, step] = 1.0
        y = x.clone()
        y[:, step] = 1.0 + 2.0**-7
        rows.view(n // 2, 2, hd)[:] = torch.stack([x, y], 1)

    def signs(rows):
        x = torch.randn(n // 2, hd, generator=g)
        rows.view(n // 2, 2, hd)[:] = torch.stack([x, -x], 1)

    pairs(k[:n], small=0, step=1)
    pairs(q[n:], small=1, step=0)
    signs(v[:n])
    signs(do[n:])
    k[n:] = torch.randn(S - n, hd, generator=g)
    q[:n] = torch.randn(n, hd, generator=g)
    q, k, v, do = (t.to(BF16) for t in (q, k, v, do))
    mask = None
    if masked:  # the same pairs, as a mask
        mask = ~torch.triu(torch.ones(S, S, dtype=torch.bool, device=DEV), 1)
    o, lse, dq, dk, dv = _call(torch.cat([q, k, v], 1).to(DEV), do.to(DEV), 1, S, 1, 1, hd, mask)

    scale = hd**-0.5
    Q, K, V, dO, O = (t.double().cpu() for t in (q, k, v, do, o))
    s = (Q @ K.t()) * scale
    s = s.masked_fill(torch.triu(torch.ones(S, S, dtype=torch.bool), 1), -math.inf)
    P = torch.softmax(s, -1)
    assert float((lse.cpu()[0, 0].double() - torch.logsumexp(s, -1)).abs().max()) < 1e-6
    dS = P * (dO @ V.t() - (dO * O).sum(-1, keepdim=True))  # delta from the rounded O, as the kernels form it
    want = {"o": (P @ V)[n:], "dq": scale * (dS @ K)[n:], "dk": scale * (dS.t() @ Q)[:n], "dv": (P.t() @ dO)[:n]}
    got = {"o": o[n:], "dq": dq[n:], "dk": dk[:n], "dv": dv[:n]}
    err = {key: float((got[key].cpu().double() - w).norm() / w.norm()) for key, w in want.items()}
    assert max(err.values()) < 0.005, err


def _hidden(kind, B, S):
    """What each query sees, and the mask that says so."""
    see = ~torch.triu(torch.ones(S, S, dtype=torch.bool), 1).repeat(B, 1, 1, 1)
    if kind in ("causal", "dropout"):
        return see, None
    see[..., S - 12 :] = False  # keys nobody sees
    if kind == "bool":
        return see, see.to(DEV)
    return see, torch.zeros(B, 1, S, S).masked_fill(~see, -math.inf).to(DEV)


@pytest.mark.parametrize("what", ["q", "k", "v", "do"])
@pytest.mark.parametrize("dtype,hd,kind,t", [
    (dtype, hd, kind, t) for dtype, hd in ((BF16, 32), (BF16, 64), (F16, 64), (F32, 32), (F32, 128))
    for kind, t in (("causal", 40), ("dropout", 40), ("bool", 40), ("additive", 40), ("bool", 66), ("additive", 66))
    if (dtype, hd, kind) != (BF16, 64, "causal")])  # its weights are rounded and zero where hidden, as in the tiles
def test_non_finite_rows_reach_only_what_sees_them(dtype, hd, kind, t, what):
    """One token's q, k, v or dO is infinite (or NaN): rows that do not see it
    are those of a clean call (float64, tolerances as elsewhere: one rounding
    of the output type), rows that do are not finite."""
    B, S, H, KV = 1, 72, 4, 2
    g = torch.Generator().manual_seed(t + hd)
    ld = (H + 2 * KV) * hd
    qkv = torch.randn(B * S, ld, generator=g).to(dtype)
    do = torch.randn(B * S, H * hd, generator=g).to(dtype)
    see, mask = _hidden(kind, B, S)
    p, key, keep = 0.0, 0, torch.ones(B, H, S, S, dtype=torch.float64)
    if kind == "dropout":
        p, key = 0.25, ops.dropout_key(5, S)
        keep = ops.dropout_mask(B * H * S * S, p, key, DEV).cpu().view(B, H, S, S).double() / (1 - p)
    bad = math.nan if what == "q" else math.inf
    dirty, ddo = qkv.clone(), do.clone()
    cols = {"q": slice(0, H * hd), "k": slice(H * hd, (H + KV) * hd), "v": slice((H + KV) * hd, ld)}
    if what == "do":
        ddo[t] = bad
    else:
        dirty[t, cols[what]] = bad
    o, _, dq, dk, dv = _call(dirty.to(DEV), ddo.to(DEV), B, S, H, KV, hd, mask, p, key)

    q, k, v = (_heads(qkv[:, cols[n]], B, S, H if n == "q" else KV, hd).clone().requires_grad_() for n in "qkv")
    K, V = k.repeat_interleave(H // KV, 1), v.repeat_interleave(H // KV, 1)
    s = ((q @ K.transpose(-1, -2)) * hd**-0.5).masked_fill(~see, -math.inf)
    oref = (torch.softmax(s, -1) * keep) @ V
    oref.backward(_heads(do, B, S, H, hd))
    rows = torch.arange(S)
    unseen = rows > t  # keys that query t does not see
    if what in ("k", "v"):
        clean_q = ~see[0, 0, :, t]
        clean_kv = {"dv": what == "v" or not bool(see[0, 0, :, t].any()), "dk": not bool(see[0, 0, :, t].any())}
        kv_rows = torch.ones(S, dtype=torch.bool)
    else:
        clean_q = rows != t
        clean_kv = {"dv": True, "dk": True}
        kv_rows = unseen | ~see[0, 0, t]
    otol, gtol = {BF16: (1e-2, 2e-2), F16: (2e-3, 5e-3), F32: (1e-5, 1e-5)}[dtype]

    def check(name, got, want, sel, tol):
        a, b = _heads(got, B, S, want.shape[1], hd)[:, :, sel], want.detach()[:, :, sel]
        assert bool(a.isfinite().all()), name
        assert float((a - b).norm()) <= tol * float(max(b.norm(), 1e-3 * want.norm())), name

    if what != "do":
        check("o", o, oref, clean_q, otol)
        dirty_o = _heads(o, B, S, H, hd)[:, :, ~clean_q]
        if what == "v" and kind != "dropout":
            assert bool((dirty_o == math.inf).all())  # positive weights of an infinite value
        elif kind != "dropout":
            assert not bool(dirty_o.isfinite().any())
    check("dq", dq, q.grad, clean_q, gtol)
    if clean_kv["dk"]:
        check("dk", dk, k.grad, kv_rows, gtol)
    if clean_kv["dv"]:
        check("dv", dv, v.grad, kv_rows, gtol)


@pytest.mark.parametrize("S", [33, 200])
@pytest.mark.parametrize("H,KV,hd", [(12, 4, 64), (16, 8, 128)])
def test_output_gradient_at_an_8_byte_offset(H, KV, hd, S):
    """The attention layer's backward takes an output gradient that is a slice
    of a flat buffer (contiguous, 8- but not 16-byte aligned) at lengths that
    are not a multiple of 64.
    bf16 outputs of weights rounded once: the gradients differ from those of an
    aligned copy by that rounding."""
    from lzhip import functional as LF

    B, d = 2, 256
    g = torch.Generator(device=DEV).manual_seed(S + hd)
    x = torch.randn(B, S, d, generator=g, device=DEV).to(BF16).requires_grad_()
    w = [(0.06 * torch.randn(n * hd, d, generator=g, device=DEV)).to(BF16).requires_grad_() for n in (H, KV, KV)]
    cos, sin = ops.rope_table(S, hd, 10000.0 ** (-torch.arange(0, hd, 2, device=DEV) / hd), BF16)
    y = LF.AttnProjFn.apply(x, *w, cos, sin, H, KV, hd**-0.5)
    flat = torch.randn(y.numel() + 4, generator=g, device=DEV).to(BF16)
    do = flat[4:].view(y.shape)
    assert do.data_ptr() % 16 == 8
    got = torch.autograd.grad(y, [x, *w], do, retain_graph=True)
    want = torch.autograd.grad(y, [x, *w], do.clone())
    for a, b in zip(got, want):
        assert float((a.double() - b.double()).norm() / b.double().norm()) < 1e-2
