"""The merges of split keys on both sides of the rule between them (a wave a
row up to three splits, a workgroup a row from four), against float64.

Bound: as in the operator's own tests, 2e-2 of the largest output in bf16 and
1e-5 in fp32."""
import math

import pytest
import torch

import coda_gqa_l

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hkv,G,Dh,Lq,Lk,dtype", [
    (256, 1, 1, 64, 1, 300, "bf16"), (171, 1, 2, 32, 1, 300, "bf16"), (128, 1, 1, 128, 2, 300, "bf16"),
    (103, 1, 1, 64, 1, 400, "bf16"), (8, 1, 4, 64, 2, 4100, "bf16"), (1, 8, 1, 64, 8, 4200, "bf16"),
    (1, 7, 8, 128, 1, 5000, "bf16"), (2, 1, 1, 64, 3, 1100, "f32"), (1, 2, 4, 128, 5, 1600, "f32"),
    (1, 1, 8, 32, 2, 2100, "f32"), (4, 1, 1, 64, 9, 4000, "f32")])
def test_against_float64(B, Hkv, G, Dh, Lq, Lk, dtype):
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    g = torch.Generator().manual_seed(B * Lk)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dt)  # noqa: E731
    q, qn, k, v = rnd(B, Hkv * G, Lq, Dh), rnd(B, Hkv * G, Lq, Dh), rnd(B, Hkv, Lk, Dh), rnd(B, Hkv, Lk, Dh)
    k[:, :, Lk // 2] *= 4  # (one split holds the largest scores)
    lam = torch.rand(B, Hkv * G, Lq, 1, generator=g).to(dt)
    got = coda_gqa_l.diff_flash_attn(*(t.cuda() for t in (q, qn, k, v, lam)), is_causal=True)  # (no weight: no norm)
    q, qn, k, v, lam = (t.double() for t in (q, qn, k, v, lam))
    k, v = k.repeat_interleave(G, 1), v.repeat_interleave(G, 1)
    vis = torch.ones(Lq, Lk, dtype=torch.bool).tril(Lk - Lq)
    a, b = (torch.softmax((x @ k.transpose(-1, -2) / math.sqrt(Dh)).masked_fill(~vis, -math.inf), -1) @ v for x in (q, qn))
    y = a - lam * b
    err = float((got.double().cpu() - y).abs().max() / y.abs().max())
    assert err <= (1e-5 if dtype == "f32" else 2e-2), err
