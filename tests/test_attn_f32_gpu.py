"""The fp32 attention kernel and the merge of split keys against float64, at
the edges of the query and key tiles and of the splits.

Bound: a score is a sum of Dh products of order 1 (error ~ sqrt(Dh) 2^-24),
its exponential carries that relative error, and the sums over Lk keys and the
norm add a few 2^-24 each: some 1e-6 of the largest output in all; 1e-5 is
held.  bf16 rows: their own rounding, 2e-2."""
import math

import pytest
import torch

import coda_gqa_l
from coda_gqa_l import ops

pytestmark = pytest.mark.gpu


def _ref(q, qn, k, v, lam, w, vis):
    q, qn, k, v, lam = (t.double() for t in (q, qn, k, v, lam))
    G = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(G, 1), v.repeat_interleave(G, 1)
    o = []
    for x in (q, qn):
        s = (x @ k.transpose(-1, -2) / math.sqrt(q.shape[-1])).masked_fill(~vis, -math.inf)
        p = torch.softmax(s, -1)
        o.append(torch.nan_to_num(p) @ v)
    y = o[0] - lam * o[1]
    return y * torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-6) * w.double()


def _close(got, ref, tol):
    err = (got.double().cpu() - ref).abs().max() / ref.abs().max()
    assert err <= tol, float(err)


@pytest.mark.parametrize("B,Hkv,G,Dh,Lq,Lk,causal,dtype", [
    (1, 1, 1, 32, 1, 1, False, "f32"), (1, 2, 2, 64, 7, 15, True, "f32"), (2, 1, 3, 128, 5, 16, False, "f32"),
    (1, 3, 4, 64, 17, 17, True, "f32"), (1, 1, 5, 32, 9, 250, True, "f32"), (2, 2, 6, 64, 3, 129, True, "f32"),
    (1, 1, 7, 128, 4, 100, False, "f32"), (1, 2, 8, 64, 33, 500, True, "f32"), (1, 1, 4, 64, 1, 5000, False, "f32"),
    (1, 2, 8, 128, 2, 4097, True, "f32"), (3, 2, 1, 32, 9, 3001, True, "f32"), (1, 4, 4, 64, 700, 1333, True, "f32"),
    (2, 8, 2, 128, 300, 300, True, "f32"), (1, 1, 4, 64, 1, 5000, False, "bf16"), (3, 2, 8, 128, 1, 777, False, "bf16"),
    (1, 1, 1, 32, 8, 9000, True, "bf16"), (1, 1, 2, 64, 3, 33000, True, "bf16")])
def test_operator_against_float64(B, Hkv, G, Dh, Lq, Lk, causal, dtype):
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    g = torch.Generator().manual_seed(Lk * 13 + Lq)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dt)  # noqa: E731
    q, qn = rnd(B, Hkv * G, Lq, Dh), rnd(B, Hkv * G, Lq, Dh)
    # rows that start on any 4-byte address: views into wider rows
    off = 1 if dtype == "f32" else 8
    k, v = rnd(B, Hkv, Lk, Dh + 16)[..., off:off + Dh], rnd(B, Hkv, Lk, Dh + 16)[..., off:off + Dh]
    lam, w = torch.rand(B, Hkv * G, Lq, 1, generator=g).to(dt), (1 + 0.1 * torch.randn(Dh, generator=g)).to(dt)
    vis = torch.ones(Lq, Lk, dtype=torch.bool)
    if causal:
        vis = vis.tril(Lk - Lq)
    dev = lambda t: torch.empty_strided(t.shape, t.stride(), dtype=t.dtype, device="cuda").copy_(t)  # noqa: E731
    kw = torch.empty(B, Hkv, Lk, Dh + 16, dtype=dt, device="cuda")
    vw = torch.empty_like(kw)
    kd, vd = kw[..., off:off + Dh], vw[..., off:off + Dh]
    kd.copy_(k)
    vd.copy_(v)
    got = coda_gqa_l.diff_flash_attn(dev(q), dev(qn), kd, vd, dev(lam), dev(w), is_causal=causal)
    _close(got, _ref(q, qn, k, v, lam, w, vis), 1e-5 if dtype == "f32" else 2e-2)


@pytest.mark.parametrize("B,Hkv,G,Dh,Lq,Lp,Lb", [(1, 2, 4, 64, 20, 37, 20), (2, 1, 8, 128, 5, 384, 21),
                                                 (1, 1, 1, 32, 1, 2048, 0), (1, 2, 2, 64, 300, 33, 300)])
def test_bounded_masks_against_float64(B, Hkv, G, Dh, Lq, Lp, Lb):
    """Prefix slots gated by `allowed` (one sequence with none visible) in
    front of the causal block."""
    g = torch.Generator().manual_seed(Lp)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    H = Hkv * G
    q, kp, vp = rnd(B, H, Lq, Dh), rnd(B, Hkv, Lp, Dh), rnd(B, Hkv, Lp, Dh)
    kb, vb = rnd(B, Hkv, max(Lb, 1), Dh)[:, :, :Lb], rnd(B, Hkv, max(Lb, 1), Dh)[:, :, :Lb]
    allowed = torch.rand(B, Lp, generator=g) < 0.5
    if Lb:
        allowed[0] = False
    ang = rnd(H, Dh // 2)
    lam, w = torch.rand(B, H, Lq, generator=g), 1 + 0.1 * rnd(Dh)
    out = torch.empty(B, H, Lq, Dh, device="cuda")
    ops.bounded_attention(
        q=q.cuda(), rope_cos=None, rope_sin=None, rope_interleaved=True, theta_cos=ang.cos().cuda(),
        theta_sin=ang.sin().cuda(), k_prefix=kp.cuda(), v_prefix=vp.cuda(), allowed=allowed.cuda(),
        k_block=kb.cuda() if Lb else None, v_block=vb.cuda() if Lb else None, lam=lam.cuda(), rms_weight=w.cuda(),
        eps=1e-6, out=out)
    c, s = ang.cos()[None, :, None], ang.sin()[None, :, None]
    qn = torch.stack([q[..., 0::2] * c - q[..., 1::2] * s, q[..., 0::2] * s + q[..., 1::2] * c], -1).flatten(-2)
    for b in range(B):
        vis = torch.cat([allowed[b].expand(Lq, Lp), torch.ones(Lq, Lb, dtype=torch.bool).tril(Lb - Lq)], 1)
        ref = _ref(q[b:b + 1], qn[b:b + 1], torch.cat([kp, kb], 2)[b:b + 1], torch.cat([vp, vb], 2)[b:b + 1],
                   lam[b:b + 1, :, :, None], w, vis)
        _close(out[b:b + 1], ref, 1e-5)
