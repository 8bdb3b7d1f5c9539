"""The kept snapshot buffers of grouped prefill: as many chunks as the longest
call so far needed, and the same results from buffers that grew."""
import pytest
import torch

import coda_gqa_l
from coda_gqa_l import state_io

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@torch.no_grad()
def test_sized_by_the_calls(dtype):
    def make():
        torch.manual_seed(3)
        return coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=32,
                                               num_landmarks_exact=8, num_landmarks_summary=8).to(DEV, dtype).eval()

    m = make()
    x = torch.randn(1, 700, 256, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).to(dtype)
    st0 = m.init_state(batch_size=1, device=DEV, dtype=dtype)
    for L, chunks in ((100, 7), (300, 19), (50, 19), (700, 44)):
        st, other = state_io.deep_copy_state(st0), state_io.deep_copy_state(st0)
        y, _ = m.prefill_chunked(x[:, :L], st, block_size=16)
        (buf,) = m._snap_cache.values()
        assert buf[0].shape[0] == buf[2].shape[0] == chunks
        z, _ = make().prefill_chunked(x[:, :L], other, block_size=16)
        assert torch.equal(y, z) and torch.equal(st.k_buf, other.k_buf) and torch.equal(st.v_buf, other.v_buf)
