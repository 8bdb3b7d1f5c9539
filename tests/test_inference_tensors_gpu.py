"""Layers built, or moved to the device, inside torch.inference_mode(): their
tensors have no version counter."""
import pytest
import torch

import coda_gqa_l

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("moved_only", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_unbounded(moved_only, dtype):
    def make():
        torch.manual_seed(4)
        return coda_gqa_l.CoDAGQA(embed_dim=512, num_heads=8, num_kv_heads=2)

    n = make().to(DEV, dtype).eval()
    m = make() if moved_only else None
    with torch.inference_mode():
        m = (m or make()).to(DEV, dtype).eval()
        p, x = torch.randn(1, 40, 512, device=DEV).to(dtype), torch.randn(1, 1, 512, device=DEV).to(dtype)
        for _ in range(2):
            out = []
            for layer in (m, n):
                y, kv = layer(p)
                out.append((y, *kv, layer(x, is_causal=False, past_key_value=kv)[0]))
            for a, b in zip(*out):
                assert torch.equal(a, b)


@pytest.mark.parametrize("B,dtype", [(1, torch.bfloat16), (70, torch.bfloat16), (2, torch.float32)])
def test_bounded_moved_inside(B, dtype):
    def make():
        torch.manual_seed(B)
        return coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16,
                                               num_landmarks_exact=8, num_landmarks_summary=8)

    m, n = make(), make().to(DEV, dtype).eval()
    with torch.inference_mode():
        m = m.to(DEV, dtype).eval()
    assert m.rope.inv_freq.is_inference()
    x = torch.randn(B, 60, 256, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).to(dtype)
    with torch.no_grad():
        out = []
        for layer in (m, n):
            torch.manual_seed(9)
            st = layer.init_state(batch_size=B, device=DEV, dtype=dtype)
            ys = [layer.prefill_chunked(x[:, :50], st, block_size=16)[0]]
            out.append(ys + [layer.step(x[:, 50 + t:51 + t], st)[0].clone() for t in range(3)] + [st.k_buf, st.v_buf])
        # (torch takes another GEMM for such weights: sums in another order)
        tol = 1e-5 if dtype == torch.float32 else 2e-2
        for a, b in zip(*out):
            assert float((a.float() - b.float()).abs().max()) <= tol * float(b.float().abs().max())
