"""CoDAGQA.forward on top of a past: the fused route (row projections, the
attention that also writes the concatenated K / V) against the module's own
linears, torch.cat and operator (a hook on one linear keeps the call there)."""
import pytest
import torch

import coda_gqa_l

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,D,H,Hkv,L,past,inter,norm", [
    (1, 512, 8, 2, 1, 1, True, "full"), (2, 512, 4, 4, 1, 15, False, "identity"), (3, 256, 8, 1, 1, 16, True, "full"),
    (1, 512, 8, 8, 8, 17, True, "full"), (2, 1024, 8, 4, 4, 255, False, "full"), (4, 512, 8, 2, 2, 513, True, "identity"),
    (1, 4096, 32, 8, 1, 4096, True, "full"), (5, 512, 4, 1, 2, 3001, False, "full"), (64, 512, 8, 1, 1, 63, True, "full"),
    (100, 256, 4, 2, 1, 40, True, "full"), (1, 512, 8, 2, 3, 50, True, "full")])
@pytest.mark.parametrize("view", [False, True])
@torch.no_grad()
def test_fused_decode_equals_module_ops(B, D, H, Hkv, L, past, inter, norm, view):
    torch.manual_seed(past + B)
    m = coda_gqa_l.CoDAGQA(embed_dim=D, num_heads=H, num_kv_heads=Hkv, rope_interleaved=inter, head_norm_mode=norm,
                           lambda_init_bias=-0.5).to(DEV, torch.bfloat16).eval()
    Dh = D // H
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(B, L, D, generator=g, device=DEV).bfloat16()
    kv = []
    for _ in range(2):
        t = torch.randn(B, Hkv, past + 5, Dh, generator=g, device=DEV).bfloat16()
        kv.append(t[:, :, 3:3 + past] if view else t[:, :, :past].contiguous())
    calls = []
    orig = m._decode
    m._decode = lambda *a: (calls.append(1), orig(*a))[1]
    ya, (ka, va) = m(x, is_causal=False, past_key_value=tuple(kv))
    assert bool(calls) == (2 * L * (H // Hkv) <= 16)
    h = m.lambda_proj.register_forward_hook(lambda *a: None)
    yb, (kb, vb) = m(x, is_causal=False, past_key_value=tuple(kv))
    h.remove()
    assert ka.shape == kb.shape and ka.stride() == kb.stride() and va.stride() == vb.stride()
    assert torch.equal(ka[:, :, :past], kb[:, :, :past]) and torch.equal(va[:, :, :past], vb[:, :, :past])
    for a, b in ((ya, yb), (ka, kb), (va, vb)):  # bf16 projections of another summation order
        assert float((a.float() - b.float()).abs().max()) <= 2e-2 * float(b.float().abs().max())
    # chained: the results are the next call's past, and causal calls stay on the general route
    n = len(calls)
    m(x, is_causal=False, past_key_value=(ka, va))
    m(x, is_causal=True, past_key_value=(ka, va))
    assert len(calls) == n + (1 if calls else 0)
