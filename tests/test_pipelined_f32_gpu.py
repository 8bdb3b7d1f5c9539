"""The fp32 prefill as bank chain + one attention launch per group of chunks
(coda_prefill_attn_chunks_f32) against the same layer chunk by chunk: states
byte-identical, heads within the fp32 order of sums (1e-5 of the largest)."""
import pytest
import torch

import coda_gqa_l
from coda_gqa_l import state_io

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D,H,Hkv,W,Me,Ms,B,L,block,group,inter", [
    (512, 8, 2, 256, 64, 64, 1, 2048, 256, None, True), (256, 4, 4, 64, 16, 16, 3, 333, 64, 2, False),
    (256, 8, 1, 32, 8, 8, 2, 100, 7, 3, True), (384, 3, 1, 40, 16, 16, 1, 200, 50, None, True),
    (512, 4, 2, 300, 32, 0, 2, 700, 128, None, False), (128, 4, 2, 16, 8, 8, 65, 70, 32, None, True),
    (160, 5, 1, 20, 0, 12, 1, 90, 16, 4, True)])
@torch.no_grad()
def test_pipelined_equals_chunk_by_chunk(D, H, Hkv, W, Me, Ms, B, L, block, group, inter):
    torch.manual_seed(L)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=D, num_heads=H, num_kv_heads=Hkv, window=W, num_landmarks_exact=Me,
                                        num_landmarks_summary=Ms, rope_interleaved=inter, lambda_init_bias=-0.5).to(DEV).eval()
    m.write_proj.weight.normal_(0, 0.7 * D ** -0.5)
    m.pipelined_group_chunks = group
    g = torch.Generator(device=DEV).manual_seed(2)
    x = torch.randn(B, L, D, generator=g, device=DEV)
    st = m.init_state(batch_size=B, device=DEV, dtype=torch.float32)
    launches = []
    orig = m._attend_chunks
    m._attend_chunks = lambda *a: (launches.append(1), orig(*a))[1]
    for part in (x, x[:, : L // 2 + 3]):  # a fresh state, then one that goes on
        other = state_io.deep_copy_state(st)
        m.pipelined_prefill = True
        ya, _ = m.prefill_chunked(part, st, block_size=block)
        n = len(launches)
        m.pipelined_prefill = False
        yb, _ = m.prefill_chunked(part, other, block_size=block)
        assert len(launches) == n
        assert float((ya - yb).abs().max()) <= 1e-5 * float(yb.abs().max())
        for f in ("k_buf", "v_buf", "allowed", "g_recent", "mem_last_exact", "_exact_v_norm", "_sum_lf_k_norm"):
            a, b = getattr(st, f), getattr(other, f)
            assert (a is None and b is None) or torch.equal(a, b), f
        assert (st.pos, st.recent_idx, st.recent_filled) == (other.pos, other.recent_idx, other.recent_filled)
    assert launches
    m.check_bank_status()
