"""coda_block_plan (the wave-wide selection) against torch's CPU topk, whose
order of ties it has to leave."""
import pytest
import torch

import coda_gqa_l  # noqa: F401
from coda_gqa_l import _hip

pytestmark = pytest.mark.gpu


def _plan(ring, head, filled, seq, block, ke, ks):
    B, L = seq.shape
    kmax = max(1, min(max(ke, ks), block))
    plan = torch.full((-(-L // block), B, kmax), -1, dtype=torch.int32, device="cuda")
    _hip.check(_hip.lib().coda_block_plan(ring.data_ptr(), head, filled, ring.shape[1], seq.data_ptr(), seq.stride(0), B,
                                          L, block, ke, ks, int(ke > 0), int(ks > 0), plan.data_ptr(), kmax,
                                          _hip.stream_of(seq)))
    return plan.cpu()


def _gates(kind, B, n, g):
    x = torch.rand(B, n, generator=g)
    if kind == "ties":  # few distinct values
        return (x * 6).floor() / 8
    if kind == "bf16":
        return torch.sigmoid(2 * x - 3).bfloat16().float()
    if kind == "equal":
        return torch.full((B, n), 0.25)
    if kind == "rising":
        return torch.arange(n).float().expand(B, n).contiguous()
    if kind == "falling":
        return -torch.arange(n).float().expand(B, n).contiguous()
    if kind == "organ":  # halves that meet: the median-of-three rule's hard order
        i = torch.arange(n)
        return torch.minimum(i, n - i).float().expand(B, n).contiguous()
    if kind == "special":
        x[:, ::7] = float("nan")
        x[:, ::5] = float("inf")
        x[:, ::3] = -0.0
        x[:, 1::3] = 0.0
    return x


@pytest.mark.parametrize("kind", ["random", "ties", "bf16", "equal", "rising", "falling", "organ", "special"])
@pytest.mark.parametrize("block,ke,ks,L", [
    (1, 1, 1, 9), (3, 8, 64, 20), (4, 2, 0, 30), (5, 3, 64, 40), (63, 8, 20, 400), (64, 8, 64, 300), (65, 8, 64, 300),
    (128, 8, 64, 1000), (256, 8, 64, 2000), (257, 256, 257, 1100), (1024, 8, 64, 3000), (1024, 8, 0, 3000),
    (4096, 8, 64, 9000), (4096, 80, 65, 9000)])
def test_plan_equals_torch_topk(kind, block, ke, ks, L):
    W, B, head = 96, 3, 17
    g = torch.Generator().manual_seed(block * 31 + L)
    seq, ring = _gates(kind, B, L, g), _gates(kind, B, W, g)
    got = _plan(ring.cuda(), head, W, seq.cuda(), block, ke, ks)
    whole = torch.cat([ring.roll(-head, 1), seq], 1)
    for c in range(got.shape[0]):
        n = min(block, L - c * block)  # the ring is full: every token evicts one
        k = min(max(ke, ks), n)
        for b in range(B):
            want = torch.topk(whole[b, c * block:c * block + n], k, sorted=False).indices
            assert got[c, b, :k].tolist() == want.tolist(), (c, b)
