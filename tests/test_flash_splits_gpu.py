"""The flash kernel with its keys over several workgroups (coda_diff_attn_fwd
with the workspace coda_attn_workspace_bytes asks for) against the same call
without a workspace (one workgroup a query block) and, where the noise queries
are given, against float64.

Bound: both forms round P to bf16 per key and the output once, in another
order of sums: 2^-8 of the output's size each way, so 2e-2 of its largest
value holds for either against the other and against float64."""
import ctypes
import math

import pytest
import torch

import coda_gqa_l  # noqa: F401
from coda_gqa_l import _hip, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _both(d, out):
    L, st = _hip.lib(), _hip.stream_of(out)
    need = ctypes.c_size_t(0)
    _hip.check(L.coda_attn_workspace_bytes(d, need))
    _hip.check(L.coda_diff_attn_fwd(d, st))
    one = out.clone()
    out.zero_()
    ws = torch.full((max(need.value, 16) + 256,), 0x7f, dtype=torch.uint8, device=DEV)
    d.workspace, d.workspace_bytes = ws.data_ptr(), need.value
    _hip.check(L.coda_diff_attn_fwd(d, st))
    assert bool((ws[need.value:] == 0x7f).all()), "written past the workspace"
    return one, out, need.value


@pytest.mark.parametrize("B,Hkv,G,Dh,Lq,Lk,causal", [
    (1, 1, 1, 64, 9, 1024, True), (1, 2, 2, 128, 33, 1601, True), (2, 1, 4, 64, 17, 1100, False),
    (1, 1, 8, 128, 5, 2500, True), (1, 2, 4, 128, 100, 1151, True), (1, 1, 4, 64, 1200, 1200, True),
    (3, 1, 8, 64, 40, 1300, False), (1, 2, 4, 64, 777, 4097, True), (1, 1, 1, 128, 65, 4000, True)])
def test_given_noise(B, Hkv, G, Dh, Lq, Lk, causal):
    g = torch.Generator(device=DEV).manual_seed(Lk)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()  # noqa: E731
    H = Hkv * G
    q, qn, k, v = rnd(B, H, Lq, Dh), rnd(B, H, Lq, Dh), rnd(B, Hkv, Lk, Dh), rnd(B, Hkv, Lk, Dh)
    lam, w = torch.rand(B, H, Lq, generator=g, device=DEV).bfloat16(), 1 + 0.1 * rnd(Dh)
    out = torch.zeros(B, H, Lq, Dh, dtype=torch.bfloat16, device=DEV)
    ones = torch.ones(H, Dh // 2, dtype=torch.bfloat16, device=DEV)
    d, keep = ops.attention_desc(q=q, rope_cos=None, rope_sin=None, rope_interleaved=True, theta_cos=ones, theta_sin=ones,
                                 k_prefix=None, v_prefix=None, allowed=None, k_block=k, v_block=v, lam=lam, rms_weight=w,
                                 eps=1e-6, out=out, causal=int(causal))
    d.q_noise, d.qn_sb, d.qn_sh, d.qn_sl = qn.data_ptr(), *qn.stride()[:3]
    one, many, need = _both(d, out)
    if Lk - (Lq // 2 if causal else 0) >= 1024 and Lq < 700:
        assert need > 0
    kk, vv = (t.double().repeat_interleave(G, 1) for t in (k, v))
    vis = torch.ones(Lq, Lk, dtype=torch.bool, device=DEV)
    vis = vis.tril(Lk - Lq) if causal else vis
    o = [torch.softmax((x.double() @ kk.transpose(-1, -2) / math.sqrt(Dh)).masked_fill(~vis, -math.inf), -1) @ vv
         for x in (q, qn)]
    y = o[0] - lam.double()[..., None] * o[1]
    y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-6) * w.double()
    for t in (one, many):
        assert float((t.double() - y).abs().max()) <= 2e-2 * float(y.abs().max())


@pytest.mark.parametrize("inter", [True, False])
@pytest.mark.parametrize("B,Hkv,G,Dh,Lq,Lp,Lb", [(1, 1, 2, 64, 64, 500, 1200), (1, 2, 4, 128, 20, 2048, 20),
                                                 (2, 1, 8, 64, 30, 96, 1500), (1, 1, 1, 128, 200, 1000, 900)])
def test_roped_queries_and_prefix(B, Hkv, G, Dh, Lq, Lp, Lb, inter):
    """RoPE and the noise rotation in the kernel, prefix visibility with a
    split that sees nothing."""
    g = torch.Generator(device=DEV).manual_seed(Lp)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()  # noqa: E731
    H = Hkv * G
    ang, th = torch.rand(Lq, Dh // 2, generator=g, device=DEV) * 6, torch.rand(H, Dh // 2, generator=g, device=DEV) * 3
    allowed = torch.rand(B, Lp, generator=g, device=DEV) < 0.5
    allowed[:, : Lp * 2 // 3] = False
    out = torch.zeros(B, H, Lq, Dh, dtype=torch.bfloat16, device=DEV)
    kv = [rnd(B, Hkv, n, Dh) for n in (Lp, Lp, Lb, Lb)]
    q, lam, w = rnd(B, H, Lq, Dh), torch.rand(B, H, Lq, generator=g, device=DEV).bfloat16(), 1 + 0.1 * rnd(Dh)
    tabs = [t.bfloat16() for t in (ang.cos(), ang.sin(), th.cos(), th.sin())]
    d, keep = ops.attention_desc(q=q, rope_cos=tabs[0], rope_sin=tabs[1], rope_interleaved=inter, theta_cos=tabs[2],
                                 theta_sin=tabs[3], k_prefix=kv[0], v_prefix=kv[1], allowed=allowed, k_block=kv[2],
                                 v_block=kv[3], lam=lam, rms_weight=w, eps=1e-6, out=out)
    one, many, need = _both(d, out)
    assert need > 0
    assert float((one.float() - many.float()).abs().max()) <= 2e-2 * float(one.float().abs().max())
