"""A token in another dtype than the state's, between tokens of the right one:
refused, the state as it was, and the steps go on as if it had not been."""
import pytest
import torch

import coda_gqa_l
from coda_gqa_l import state_io

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B", [1, 20])
@pytest.mark.parametrize("state", [torch.float32, torch.bfloat16])
@torch.no_grad()
def test_other_dtype_between_tokens(B, state):
    torch.manual_seed(B)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16, num_landmarks_exact=8,
                                        num_landmarks_summary=8).to(DEV, state).eval()
    st = m.init_state(batch_size=B, device=DEV, dtype=state)
    x = torch.randn(B, 60, 256, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
    m.prefill_chunked(x[:, :50].to(state), st, block_size=16, return_outputs=False)
    st2 = state_io.deep_copy_state(st)
    other = torch.bfloat16 if state == torch.float32 else torch.float32
    for t in range(50, 53):
        a = m.step(x[:, t:t + 1].to(state), st)[0].clone()
        pos, k = st.pos, st.k_buf.clone()
        if t == 51:
            with pytest.raises((RuntimeError, TypeError)):
                m.step(x[:, t:t + 1].to(other), st)
            torch.cuda.synchronize()
            assert st.pos == pos and torch.equal(st.k_buf, k)
        assert torch.equal(a, m.step(x[:, t:t + 1].to(state), st2)[0])
    assert torch.equal(st.k_buf, st2.k_buf) and torch.equal(st.v_buf, st2.v_buf)
