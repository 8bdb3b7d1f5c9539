"""A RoPE module of the user's own in a layer's place, without the buffer that
the kernels could read: every call takes its tables from the module."""
import pytest
import torch

import coda_gqa_l

pytestmark = pytest.mark.gpu
DEV = "cuda"


class Rope(torch.nn.Module):
    def __init__(self, half, base):
        super().__init__()
        self.half, self.base = half, base

    def forward(self, *, seq_len, offset, device, dtype):
        inv = 1.0 / (self.base ** (torch.arange(0, 2 * self.half, 2, device=device).float() / (2 * self.half)))
        f = torch.arange(offset, offset + seq_len, device=device).float()[:, None] * inv[None]
        return f.cos().to(dtype), f.sin().to(dtype)


@pytest.mark.parametrize("B,dtype", [(2, torch.bfloat16), (70, torch.bfloat16), (2, torch.float32)])
@torch.no_grad()
def test_bounded(B, dtype):
    def make():
        torch.manual_seed(B)
        return coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16,
                                               num_landmarks_exact=8, num_landmarks_summary=8).to(DEV, dtype).eval()

    x = torch.randn(B, 60, 256, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).to(dtype)

    def run(m):
        torch.manual_seed(9)
        st = m.init_state(batch_size=B, device=DEV, dtype=dtype)
        ys = [m.prefill_chunked(x[:, :5], st, block_size=16)[0]] + [m.step(x[:, 5 + t:6 + t], st)[0].clone() for t in range(2)]
        ys.append(m.prefill_chunked(x[:, 7:50], st, block_size=16)[0])
        return ys + [m.step(x[:, 50 + t:51 + t], st)[0].clone() for t in range(4)] + [st.k_buf, st.v_buf]

    for base in (1e4, 500.0):
        m, n = make(), make()
        m.rope = Rope(32, base)
        n.rope.inv_freq = (1.0 / (base ** (torch.arange(0, 64, 2, device=DEV).float() / 64)))
        # (projections of another route: sums in another order)
        tol = 1e-5 if dtype == torch.float32 else 3e-2
        for a, b in zip(run(m), run(n)):
            assert float((a.float() - b.float()).abs().max()) <= tol * float(b.float().abs().max())


@torch.no_grad()
def test_unbounded():
    torch.manual_seed(4)
    m = coda_gqa_l.CoDAGQA(embed_dim=512, num_heads=8, num_kv_heads=2).to(DEV, torch.bfloat16).eval()
    p, x = torch.randn(1, 40, 512, device=DEV).bfloat16(), torch.randn(1, 1, 512, device=DEV).bfloat16()
    m.rope.inv_freq = 1.0 / (1e4 ** (torch.arange(0, 64, 2, device=DEV).float() / 64))
    y, kv = m(p)
    want = (y, m(x, is_causal=False, past_key_value=kv)[0])
    m.rope = Rope(32, 1e4)
    y, kv = m(p)
    for a, b in zip((y, m(x, is_causal=False, past_key_value=kv)[0]), want):
        assert torch.equal(a, b)
