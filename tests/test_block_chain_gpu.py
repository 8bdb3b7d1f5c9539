"""The chunk chain in one launch (coda_block_write_chain) against one call a
chunk (coda_block_write_snapshot) and against the four-kernel update, which
shares no code with it past the candidate rows: states, snapshots and ring,
bit for bit."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(monkeypatch, how, B, H, Hkv, W, Me, Ms, blk, L, warm, dtype, ke, ks, seed=5):
    """State after a warm-up prompt of `warm` tokens, then L tokens chunk by
    chunk through `how`; snapshots (n, ...) for chain and single."""
    import coda_gqa_l
    from coda_gqa_l import _hip
    torch.manual_seed(seed)
    Dh = 128 if H * 128 <= 1024 else 64
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=H * Dh, num_heads=H, num_kv_heads=Hkv, window=W,
                                        num_landmarks_exact=Me, num_landmarks_summary=Ms,
                                        exact_candidates_per_block=ke, summary_candidates_per_block=ks)
    m = m.to(DEV, dtype).eval()
    st = m.init_state(batch_size=B, device=DEV, dtype=dtype)
    g = torch.Generator(device=DEV).manual_seed(seed)
    if warm:
        m.prefill_chunked(torch.randn(B, warm, m.embed_dim, generator=g, device=DEV).to(dtype), st, block_size=blk)
    k, v = (torch.randn(B, L, Hkv, Dh, generator=g, device=DEV).to(dtype).permute(0, 2, 1, 3) for _ in range(2))
    gates = torch.rand(B, L, generator=g, device=DEV)
    plan, kmax, do_e, do_s = m._plan_candidates(st, gates, L, blk)
    ws = m._block_workspace(st, kmax)
    eta = m._eta_f32(torch.device(DEV), dtype) if Ms else None
    head, filled = (int(st.recent_idx) if st.recent_filled >= W else 0), int(st.recent_filled)
    n, S = -(-L // blk), Me + Ms
    snaps = (torch.zeros(n, B, Hkv, S, Dh, dtype=dtype, device=DEV), torch.zeros(n, B, Hkv, S, Dh, dtype=dtype, device=DEV),
             torch.zeros(n, B, S, dtype=torch.uint8, device=DEV))
    if how == "four":
        monkeypatch.setenv("CODA_BLOCK_FUSED", "0")
    if how == "chain":
        ring = (ctypes.c_int * 2)()
        _hip.check(_hip.lib().coda_block_write_chain(
            m._bank_desc(st, eta, None, None), k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(1), k.stride(2),
            gates.data_ptr(), gates.stride(0), L, blk, 0, n, head, filled, int(st.pos), plan.data_ptr(), kmax,
            ke if do_e else 0, ks if do_s else 0, ws.data_ptr(), ws.numel(), snaps[0].data_ptr(), snaps[1].data_ptr(),
            snaps[2].data_ptr(), snaps[0][0].numel(), snaps[2][0].numel(), ring, _hip.stream_of(k)))
        head, filled = int(ring[0]), int(ring[1])
    else:
        for c in range(n):
            t = slice(c * blk, min(L, (c + 1) * blk))
            snap = tuple(s[c] for s in snaps) if how == "single" else None
            head, filled = m._write_block(st, k_blk=k[:, :, t], v_blk=v[:, :, t], g_blk=gates[:, t],
                                          pos0=int(st.pos) + c * blk, ring_head=head, ring_filled=filled,
                                          plan_c=plan[c], kmax=kmax, do_e=do_e, do_s=do_s, workspace=ws, eta=eta,
                                          snap=snap)
    torch.cuda.synchronize()
    m.check_bank_status()
    monkeypatch.delenv("CODA_BLOCK_FUSED", raising=False)
    state = [st.k_buf, st.v_buf, st.allowed, st.g_recent, st.mem_last_exact, st._exact_v_norm, st._sum_lf_k_norm]
    return [x for x in state if x is not None], snaps, (head, filled)


@torch.no_grad()
@pytest.mark.parametrize("B,H,Hkv,W,Me,Ms,blk,L,warm,dtype,ke,ks", [
    (1, 8, 8, 64, 64, 64, 64, 64 * 5 + 17, 64, torch.bfloat16, 8, 64),     # slots unused: tied LRU keys
    (2, 8, 2, 100, 33, 45, 70, 70 * 4 + 3, 500, torch.bfloat16, 8, 64),    # odd sizes, few candidates in the last chunk
    (3, 4, 1, 48, 130, 70, 200, 600, 300, torch.bfloat16, 64, 33),         # a chunk longer than the ring, > 64 slots
    (5, 8, 8, 64, 16, 0, 32, 96, 200, torch.float32, 5, 8),                # exact alone, fp32
    (1, 16, 4, 64, 0, 40, 64, 200, 200, torch.float32, 8, 64),             # summary alone
    (40, 8, 8, 32, 64, 64, 32, 96, 64, torch.bfloat16, 8, 32),             # more pairs than CUs: one workgroup a head
    (1, 4, 2, 16, 24, 24, 16, 16 * 70, 32, torch.bfloat16, 4, 16),         # more chunks than a launch takes
])
def test_chain_is_the_chunks(monkeypatch, B, H, Hkv, W, Me, Ms, blk, L, warm, dtype, ke, ks):
    args = (B, H, Hkv, W, Me, Ms, blk, L, warm, dtype, ke, ks)
    want, snaps1, ring1 = _run(monkeypatch, "single", *args)
    got, snaps, ring = _run(monkeypatch, "chain", *args)
    four, _, ring4 = _run(monkeypatch, "four", *args)
    assert ring == ring1 == ring4
    for i, (a, b, c) in enumerate(zip(got, want, four)):
        assert torch.equal(a, b), f"state {i}: chain and single calls differ"
        assert torch.equal(a, c), f"state {i}: chain and the four-kernel update differ"
    for i, (a, b) in enumerate(zip(snaps, snaps1)):
        assert torch.equal(a, b), f"snapshot {i} differs"


@torch.no_grad()
@pytest.mark.parametrize("B,Hkv,W,Me,Ms,filled,blk,dtype", [
    (1, 1, 16, 8, 8, 0, 1, torch.bfloat16), (2, 3, 300, 33, 45, 17, 283, torch.bfloat16),
    (1, 2, 256, 0, 130, 100, 37, torch.float32), (3, 2, 64, 150, 0, 0, 64, torch.float32)])
def test_ring_write_with_snapshot(B, Hkv, W, Me, Ms, filled, blk, dtype):
    """coda_block_ring_snapshot: the ring of coda_block_write, the banks
    copied and untouched; a chunk that evicts is refused."""
    import coda_gqa_l
    from coda_gqa_l import _hip
    Dh, S = 64, Me + Ms
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=Hkv * Dh, num_heads=Hkv, num_kv_heads=Hkv, window=W,
                                        num_landmarks_exact=Me, num_landmarks_summary=Ms).to(DEV, dtype).eval()
    g = torch.Generator(device=DEV).manual_seed(3)
    states = []
    for _ in range(2):
        st = m.init_state(batch_size=B, device=DEV, dtype=dtype)
        g.manual_seed(3)
        st.k_buf.copy_(torch.randn(st.k_buf.shape, generator=g, device=DEV))
        st.v_buf.copy_(torch.randn(st.k_buf.shape, generator=g, device=DEV))
        st.allowed[:, W:] = torch.rand(B, S, generator=g, device=DEV) < 0.5
        states.append(st)
    k, v = (torch.randn(B, blk, Hkv, Dh, generator=g, device=DEV).to(dtype).permute(0, 2, 1, 3) for _ in range(2))
    gates = torch.rand(B, blk, generator=g, device=DEV)
    eta = m._eta_f32(torch.device(DEV), dtype) if Ms else None
    kw = dict(k_blk=k, v_blk=v, g_blk=gates, pos0=filled, ring_head=0, ring_filled=filled, plan_c=None, kmax=1,
              do_e=False, do_s=False, workspace=None, eta=eta)
    snap = (torch.zeros(B, Hkv, S, Dh, dtype=dtype, device=DEV), torch.zeros(B, Hkv, S, Dh, dtype=dtype, device=DEV),
            torch.full((B, S), 7, dtype=torch.uint8, device=DEV))
    want = [states[0].k_buf[:, :, W:].clone(), states[0].v_buf[:, :, W:].clone(), states[0].allowed[:, W:].to(torch.uint8)]
    assert m._write_block(states[0], snap=snap, **kw) == m._write_block(states[1], **kw)
    for a, b in zip(snap, want):
        assert torch.equal(a, b)
    for f in ("k_buf", "v_buf", "allowed", "g_recent"):
        assert torch.equal(getattr(states[0], f), getattr(states[1], f)), f
    rc = _hip.lib().coda_block_ring_snapshot(
        m._bank_desc(states[0], eta, None, None), k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(1), k.stride(2),
        gates.data_ptr(), gates.stride(0), blk, W - blk + 1, snap[0].data_ptr(), snap[1].data_ptr(), snap[2].data_ptr(),
        _hip.stream_of(k))
    assert rc not in (_hip.CODA_OK, _hip.CODA_EUNSUP)
