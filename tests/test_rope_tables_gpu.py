"""The RoPE tables of prompts: the same bits as the module's, for every buffer
type, and anew when inv_freq changes."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@torch.no_grad()
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("inv", [torch.bfloat16, torch.float32])
def test_cached_rows_are_the_table(dtype, inv):
    import coda_gqa_l
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=128, num_heads=2, num_kv_heads=1, window=16, num_landmarks_exact=8,
                                        num_landmarks_summary=8).to(DEV).eval()
    m.rope.inv_freq = m.rope.inv_freq.to(inv)

    def check(p0, L):
        for got, want in zip(m._rope_tables(p0, L, torch.device(DEV), dtype),
                             m.rope(seq_len=L, offset=p0, device=torch.device(DEV), dtype=dtype)):
            assert got.shape == want.shape and got.is_contiguous() and torch.equal(got, want)

    for p0, L in ((0, 1), (7, 300), (4095, 2), (3, 4093), (5000, 1999), (65535, 1), (65500, 100), (1 << 20, 5)):
        check(p0, L)
    m.rope.inv_freq.mul_(0.5)  # in place
    check(9, 64)
    m.rope.inv_freq = m.rope.inv_freq * 3  # another buffer
    check(9, 64)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        check(11, 5)
    torch.cuda.synchronize()
