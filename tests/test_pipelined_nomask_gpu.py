"""mask_unused_memory=False: the unused slots of a ring that is still filling
are attended to (zero keys and values), chunk by chunk and pipelined alike."""
import pytest
import torch

import coda_gqa_l
from coda_gqa_l import state_io

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("L", [150, 500])
@torch.no_grad()
def test_pipelined_equals_chunk_by_chunk(L):
    torch.manual_seed(1)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=512, num_heads=4, num_kv_heads=2, window=128, num_landmarks_exact=32,
                                        num_landmarks_summary=32, mask_unused_memory=False).to(DEV, torch.bfloat16).eval()
    x = torch.randn(2, L, 512, generator=torch.Generator(device=DEV).manual_seed(3), device=DEV).bfloat16()
    st = m.init_state(batch_size=2, device=DEV, dtype=torch.bfloat16)
    for _ in range(2):  # a fresh state, then one that goes on
        other = state_io.deep_copy_state(st)
        m.pipelined_prefill = True
        ya, _ = m.prefill_chunked(x, st, block_size=64)
        m.pipelined_prefill = False
        yb, _ = m.prefill_chunked(x, other, block_size=64)
        assert float((ya - yb).float().abs().max()) <= 2e-2 * float(yb.float().abs().max())
        assert torch.equal(st.k_buf, other.k_buf) and torch.equal(st.v_buf, other.v_buf)
