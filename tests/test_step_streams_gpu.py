"""Steps of one state on two streams in turn, each waiting for the other, with
allocations in between that take any memory given back too early: the same
tokens as on one stream."""
import pytest
import torch

import coda_gqa_l
from coda_gqa_l import state_io

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,dtype", [(2, torch.bfloat16), (70, torch.bfloat16), (2, torch.float32)])
@torch.no_grad()
def test_streams_in_turn(B, dtype):
    torch.manual_seed(B)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16, num_landmarks_exact=8,
                                        num_landmarks_summary=8).to(DEV, dtype).eval()
    st = m.init_state(batch_size=B, device=DEV, dtype=dtype)
    x = torch.randn(B, 70, 256, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).to(dtype)
    m.prefill_chunked(x[:, :50], st, block_size=16, return_outputs=False)
    st2 = state_io.deep_copy_state(st)
    want = [m.step(x[:, t:t + 1], st2)[0].clone() for t in range(50, 70)]
    torch.cuda.synchronize()
    streams, last, got = [torch.cuda.Stream(), torch.cuda.Stream()], None, []
    for t in range(50, 70):
        s = streams[t // 3 % 2]
        if last is not None:
            s.wait_stream(last)
        with torch.cuda.stream(s):
            y, _ = m.step(x[:, t:t + 1], st)
            got.append(y)
            assert m._fast["stream"] == s.cuda_stream
        with torch.cuda.stream(streams[1 - t // 3 % 2]):
            junk = [torch.full((1 << n,), float("nan"), device=DEV) for n in range(8, 18)]
            del junk
        last = s
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    assert torch.equal(st.k_buf, st2.k_buf) and torch.equal(st.v_buf, st2.v_buf)
