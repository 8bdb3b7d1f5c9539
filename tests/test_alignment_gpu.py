"""Activations that are contiguous but start off a 16-byte address: the same
outputs, bit for bit, as from an aligned copy."""
import pytest
import torch

import coda_gqa_l
from coda_gqa_l import state_io

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _off(x):
    flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=DEV)
    flat[1:].copy_(x.reshape(-1))
    y = flat[1:].view(x.shape)
    assert y.is_contiguous() and y.data_ptr() % 16
    return y


@pytest.mark.parametrize("B,dtype", [(1, torch.bfloat16), (70, torch.bfloat16), (2, torch.float32)])
@pytest.mark.parametrize("steady", [True, False])
@torch.no_grad()
def test_step(B, dtype, steady):
    torch.manual_seed(B)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16, num_landmarks_exact=8,
                                        num_landmarks_summary=8).to(DEV, dtype).eval()
    st = m.init_state(batch_size=B, device=DEV, dtype=dtype)
    x = torch.randn(B, 60, 256, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).to(dtype)
    m.prefill_chunked(x[:, :50 if steady else 9], st, block_size=16, return_outputs=False)
    st2 = state_io.deep_copy_state(st)
    for t in range(2):
        xt = x[:, 50 + t:51 + t].contiguous()
        assert torch.equal(m.step(_off(xt), st)[0], m.step(xt, st2)[0])
    assert torch.equal(st.k_buf, st2.k_buf) and torch.equal(st.v_buf, st2.v_buf)


@torch.no_grad()
def test_unbounded_decode():
    torch.manual_seed(4)
    m = coda_gqa_l.CoDAGQA(embed_dim=512, num_heads=8, num_kv_heads=2).to(DEV, torch.bfloat16).eval()
    x = torch.randn(2, 1, 512, device=DEV).bfloat16()
    kv = tuple(torch.randn(2, 2, 90, 64, device=DEV).bfloat16() for _ in range(2))
    (ya, a), (yb, b) = (m(t, is_causal=False, past_key_value=kv) for t in (_off(x), x))
    assert torch.equal(ya, yb) and torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
