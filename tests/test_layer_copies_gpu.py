"""A layer that has run can be copied and saved whole, and the copy computes
what the layer does: nothing that a layer keeps between calls travels."""
import copy
import io

import pytest
import torch

import coda_gqa_l

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _saved(m):
    f = io.BytesIO()
    torch.save(m, f)
    f.seek(0)
    return torch.load(f, weights_only=False)


@pytest.mark.parametrize("again", [copy.deepcopy, _saved])
@torch.no_grad()
def test_unbounded(again):
    torch.manual_seed(4)
    m = coda_gqa_l.CoDAGQA(embed_dim=512, num_heads=8, num_kv_heads=2).to(DEV, torch.bfloat16).eval()
    p, x = torch.randn(1, 40, 512, device=DEV).bfloat16(), torch.randn(1, 1, 512, device=DEV).bfloat16()

    def run(m):
        y, kv = m(p)
        return y, m(x, is_causal=False, past_key_value=kv)[0]

    want = run(m)
    for a, b in zip(run(again(m)), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("again", [copy.deepcopy, _saved])
@pytest.mark.parametrize("B,dtype", [(1, torch.bfloat16), (70, torch.bfloat16), (2, torch.float32)])
@torch.no_grad()
def test_bounded(again, B, dtype):
    torch.manual_seed(B)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16, num_landmarks_exact=8,
                                        num_landmarks_summary=8).to(DEV, dtype).eval()
    x = torch.randn(B, 60, 256, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).to(dtype)

    def run(m):
        torch.manual_seed(9)
        st = m.init_state(batch_size=B, device=DEV, dtype=dtype)
        ys = [m.prefill_chunked(x[:, :50], st, block_size=16)[0]]
        return ys + [m.step(x[:, 50 + t:51 + t], st)[0] for t in range(3)] + [st.k_buf, st.v_buf]

    want = run(m)
    n = again(m)
    assert n.state_dict().keys() == m.state_dict().keys() and not n.training
    n.o_proj.weight.mul_(1)  # (its parameters are its own)
    for a, b in zip(run(n), want):
        assert torch.equal(a, b)
