"""fp32 prefill whose last group holds one chunk, with keys enough and
workgroups few enough that a launch of its own would split the keys: the
grouped launch must not (its splits would need a workspace, and their merge
the chunk's own rows)."""
import ctypes

import pytest
import torch

import coda_gqa_l
from coda_gqa_l import _hip, ops, state_io

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("H,Hkv,D,W,bank,block,L,group", [
    (4, 1, 256, 512, 128, 256, 700, None), (2, 2, 256, 512, 128, 256, 700, None), (4, 1, 256, 768, 64, 128, 2100, 1),
    (1, 1, 64, 1024, 32, 64, 1270, 3)])
@torch.no_grad()
def test_equals_chunk_by_chunk(H, Hkv, D, W, bank, block, L, group):
    torch.manual_seed(L)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=D, num_heads=H, num_kv_heads=Hkv, window=W, num_landmarks_exact=bank,
                                        num_landmarks_summary=bank, lambda_init_bias=-0.5).to(DEV).eval()
    m.pipelined_group_chunks = group
    g = torch.Generator(device=DEV).manual_seed(2)
    st = m.init_state(batch_size=1, device=DEV, dtype=torch.float32)
    m.prefill_chunked(torch.randn(1, W + block, D, generator=g, device=DEV), st, block_size=block, return_outputs=False)
    other = state_io.deep_copy_state(st)
    x = torch.randn(1, L, D, generator=g, device=DEV)
    ones = []
    orig = m._attend_chunks
    m._attend_chunks = lambda *a: (ones.append(a[14] - a[13] == 1), orig(*a))[1]
    ya, _ = m.prefill_chunked(x, st, block_size=block)
    assert any(ones), "no group of one chunk"
    m.pipelined_prefill = False
    yb, _ = m.prefill_chunked(x, other, block_size=block)
    # (fp32 sums in another order)
    assert float((ya - yb).abs().max()) <= 1e-5 * float(yb.abs().max())
    for f in ("k_buf", "v_buf", "allowed", "g_recent", "mem_last_exact", "_exact_v_norm", "_sum_lf_k_norm"):
        assert torch.equal(getattr(st, f), getattr(other, f)), f


@pytest.mark.parametrize("workspace", [0, 1 << 24])
@torch.no_grad()
def test_one_chunk_call_with_and_without_workspace(workspace):
    """The library call itself for chunk 2 of a call: its own rows alone are
    written, whatever workspace the descriptor names."""
    B, H, Hkv, Dh, blk, L, W, S = 1, 4, 1, 64, 256, 700, 512, 256
    g = torch.Generator(device=DEV).manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    q, k, v = rnd(B, H, L, Dh), rnd(B, Hkv, L, Dh), rnd(B, Hkv, L, Dh)
    kp, vp, lam, th = rnd(B, Hkv, S, Dh), rnd(B, Hkv, S, Dh), torch.rand(B, H, L, generator=g, device=DEV), rnd(H, Dh // 2)
    ang = rnd(L, Dh // 2)
    cos, sin, out = ang.cos(), ang.sin(), torch.full((B, L, H, Dh), 7.0, device=DEV)
    kw = dict(rope_interleaved=True, theta_cos=th.cos(), theta_sin=th.sin(), k_prefix=kp, v_prefix=vp, allowed=None,
              rms_weight=None, eps=1e-6)
    d, keep = ops.attention_desc(q=q, rope_cos=cos, rope_sin=sin, k_block=k, v_block=v, lam=lam,
                                 out=out.permute(0, 2, 1, 3), **kw)
    ws = torch.empty(max(workspace, 1), dtype=torch.uint8, device=DEV)
    d.workspace, d.workspace_bytes = (ws.data_ptr(), workspace) if workspace else (None, 0)
    _hip.check(_hip.lib().coda_prefill_attn_chunks_f32(ctypes.byref(d), 1, 2, blk, L, W, 0, 0, _hip.stream_of(q)))
    t0 = 2 * blk
    want = torch.empty(B, L - t0, H, Dh, device=DEV)
    ops.bounded_attention(q=q[:, :, t0:], rope_cos=cos[t0:], rope_sin=sin[t0:], k_block=k[:, :, t0 - W:],
                          v_block=v[:, :, t0 - W:], lam=lam[:, :, t0:], out=want.permute(0, 2, 1, 3), **kw)
    assert bool((out[:, :t0] == 7).all())
    assert float((out[:, t0:] - want).abs().max()) <= 1e-5 * float(want.abs().max())
