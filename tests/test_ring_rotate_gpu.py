"""coda_ring_rotate (a full ring into time order, in place) against torch.roll,
byte for byte, at the edges of its register strips and past them."""
import pytest
import torch

import coda_gqa_l  # noqa: F401
from coda_gqa_l import _hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W,head,Dh,Hkv,B", [
    (2, 1, 32, 1, 1), (63, 62, 64, 2, 1), (64, 1, 128, 3, 2), (65, 33, 64, 1, 2), (128, 127, 128, 2, 1),
    (129, 5, 32, 2, 3), (256, 100, 128, 8, 1), (257, 256, 64, 2, 1), (512, 511, 128, 1, 2), (513, 200, 32, 1, 1),
    (2048, 77, 64, 1, 2), (2049, 1000, 64, 1, 1)])
def test_ring_rotate_equals_roll(W, head, Dh, Hkv, B, dtype):
    g = torch.Generator().manual_seed(W * 7 + head)
    bank = 5
    k = torch.randn(B, Hkv, W + bank, Dh, generator=g).to(dtype).cuda()
    v = torch.randn(B, Hkv, W + bank, Dh, generator=g).to(dtype).cuda()
    gates = torch.rand(B, W, generator=g).cuda()
    allowed = torch.ones(B, W + bank, dtype=torch.bool, device="cuda")
    want = [torch.cat([t[:, :, :W].roll(-head, 2), t[:, :, W:]], 2) for t in (k, v)] + [gates.roll(-head, 1)]
    d = _hip.BankDesc()
    d.dtype, d.B, d.Hkv, d.Dh, d.W, d.Me, d.Ms, d.lf = _hip.dtype_code(dtype), B, Hkv, Dh, W, bank, 0, Dh // 2
    d.active_exact = bank
    d.k_buf, d.v_buf, d.allowed, d.g_recent = k.data_ptr(), v.data_ptr(), allowed.data_ptr(), gates.data_ptr()
    need = B * Hkv * W * Dh * 2 * k.element_size() + B * W * 4
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    _hip.check(_hip.lib().coda_ring_rotate(d, head, ws.data_ptr(), need, _hip.stream_of(k)))
    for got, ref in zip((k, v, gates), want):
        assert torch.equal(got, ref)
