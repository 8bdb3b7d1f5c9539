"""coda_diff_attn_fwd in fp32 with few queries and many keys, the workspace of
its key splits missing or too small: one launch without splits, the same
result up to the order of fp32 sums."""
import ctypes
import math

import pytest
import torch

from coda_gqa_l import _hip

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("H,Hkv,Lq,Lk,Dh", [(4, 1, 1, 5000, 64), (2, 2, 3, 1100, 32), (8, 1, 40, 4097, 128)])
def test_without_workspace(H, Hkv, Lq, Lk, Dh):
    g = torch.Generator(device=DEV).manual_seed(Lk)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    q, qn, k, v, lam = rnd(1, H, Lq, Dh), rnd(1, H, Lq, Dh), rnd(1, Hkv, Lk, Dh), rnd(1, Hkv, Lk, Dh), rnd(1, H, Lq)
    L, outs = _hip.lib(), []
    for room in (None, 64, -1):
        out = torch.full((1, H, Lq, Dh), 7.0, device=DEV)
        d = _hip.AttnDesc()
        d.dtype, d.B, d.H, d.Hkv, d.Lq, d.Dh = _hip.CODA_F32, 1, H, Hkv, Lq, Dh
        d.q, (d.q_sb, d.q_sh, d.q_sl) = q.data_ptr(), q.stride()[:3]
        d.q_noise, (d.qn_sb, d.qn_sh, d.qn_sl) = qn.data_ptr(), qn.stride()[:3]
        d.kb, d.vb, d.Lb, (d.b_sb, d.b_sh, d.b_sl) = k.data_ptr(), v.data_ptr(), Lk, k.stride()[:3]
        d.lam, (d.lam_sb, d.lam_sh, d.lam_sl) = lam.data_ptr(), lam.stride()
        d.eps, d.sm_scale, d.causal = 1e-6, 1 / math.sqrt(Dh), 1
        d.out, (d.o_sb, d.o_sh, d.o_sl) = out.data_ptr(), out.stride()[:3]
        need = ctypes.c_size_t(0)
        _hip.check(L.coda_attn_workspace_bytes(d, need))
        assert need.value > 64, "the shape does not split"
        n = need.value if room == -1 else room or 0
        ws = torch.empty(max(n, 1), dtype=torch.uint8, device=DEV)
        d.workspace, d.workspace_bytes = (ws.data_ptr(), n) if n else (None, 0)
        _hip.check(L.coda_diff_attn_fwd(d, _hip.stream_of(q)))
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    assert float((outs[0] - outs[2]).abs().max()) <= 1e-5 * float(outs[2].abs().max())
