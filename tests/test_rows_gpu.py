"""coda_linear_rows over coda_rows_pack's tiles (the few-row kernels, straight
from memory and through LDS) against float64, at the edges of their token
blocks, feature blocks and K splits; and the layer's step at the sizes whose
route depends on them.

Bound: fp32 accumulation of D products of order D^-1/2 (error well below
1e-6 of the result's spread), then one rounding: 2^-9 of the element in bf16
(half a unit of its 8 bits), 2^-24 sqrt(D) in fp32."""
import pytest
import torch

import coda_gqa_l
from coda_gqa_l import _hip, state_io

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,D,bias", [
    (1, 1, 64, False), (3, 17, 64, True), (16, 64, 128, False), (17, 50, 192, True), (1, 777, 512, False),
    (31, 33, 1024, True), (32, 48, 2048, False), (33, 4096, 320, False), (64, 100, 2048, True), (65, 63, 1088, False),
    (100, 8200, 256, True), (128, 6184, 2048, False), (127, 4100, 4096, True), (64, 8193, 1024, False),
    (48, 12300, 1024, True), (20, 8208, 6144, False)])
def test_linear_rows_against_float64(M, N, D, bias, dtype):
    g = torch.Generator(device=DEV).manual_seed(M * 1000 + N)
    w = (torch.randn(N, D, generator=g, device=DEV) * D ** -0.5).to(dtype)
    x = torch.randn(M, D + 8, generator=g, device=DEV).to(dtype)[:, :D]  # rows farther apart than their length
    b = torch.randn(N, generator=g, device=DEV) if bias else None
    code, st, L = _hip.dtype_code(dtype), _hip.stream_of(x), _hip.lib()
    tiles = torch.empty(-(-N // 64) * 64, D, device=DEV, dtype=dtype)
    _hip.check(L.coda_rows_pack(code, w.data_ptr(), N, D, D, tiles.data_ptr(), st))
    ld = N + (-N) % 4 + 4
    out = torch.full((M + 1, ld), 7.0, device=DEV, dtype=dtype)
    _hip.check(L.coda_linear_rows(code, x.data_ptr(), x.stride(0), M, tiles.data_ptr(), N, D, _hip.ptr(b), out.data_ptr(),
                                  ld, st))
    ref = x.double() @ w.double().t() + (b.double() if bias else 0)
    err = (out[:M, :N].double() - ref).abs()
    tol = 2.0 ** -8 * ref.abs() + 1e-5 if dtype == torch.bfloat16 else 1e-6 * ref.abs() + 1e-5
    assert bool((err <= tol).all()), float((err - tol).max())
    assert bool((out[M:] == 7).all()) and bool((out[:, N:] == 7).all()), "written past the rows or features"


@pytest.mark.parametrize("B,D,H,Hkv,dtype", [(1, 512, 8, 2, "f32"), (32, 256, 4, 2, "f32"), (33, 256, 4, 2, "f32"),
                                             (3, 320, 5, 5, "bf16"), (65, 512, 4, 1, "bf16"), (128, 1024, 8, 4, "bf16"),
                                             (129, 512, 8, 8, "bf16")])
@torch.no_grad()
def test_step_equals_the_linears_route(B, D, H, Hkv, dtype):
    """step() against the same step through the module's own linears (a hook
    on one of them keeps it off the row kernels): the token's K / V rows and
    the output within rounding, the banks (decided by older tokens) equal."""
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    torch.manual_seed(B + D)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=D, num_heads=H, num_kv_heads=Hkv, window=32, num_landmarks_exact=16,
                                        num_landmarks_summary=16).to(DEV, dt).eval()
    st = m.init_state(batch_size=B, device=DEV, dtype=dt)
    g = torch.Generator(device=DEV).manual_seed(9)
    m.prefill_chunked(torch.randn(B, 70, D, generator=g, device=DEV).to(dt), st, block_size=32, return_outputs=False)
    st2 = state_io.deep_copy_state(st)
    x = torch.randn(B, 1, D, generator=g, device=DEV).to(dt)
    ya, _ = m.step(x, st)
    hook = [m.lambda_proj.register_forward_hook(lambda *a: None), m.o_proj.register_forward_hook(lambda *a: None)]
    if B <= 64 and dt == torch.bfloat16:  # (this route needs no plain linears)
        m._fused_front_ok, m._step_fast = lambda x: False, lambda *a: None
    yb, _ = m.step(x, st2)
    for h in hook:
        h.remove()
    tol = 1e-5 if dtype == "f32" else 2e-2
    for a, b in ((ya, yb), (st.k_buf, st2.k_buf), (st.v_buf, st2.v_buf)):
        assert float((a.double() - b.double()).abs().max()) <= tol * float(b.double().abs().max())
    assert torch.equal(st.k_buf[:, :, 32:], st2.k_buf[:, :, 32:]) and torch.equal(st.allowed, st2.allowed)
    assert torch.equal(st.mem_last_exact, st2.mem_last_exact)


@torch.no_grad()
def test_weights_off_16_byte_addresses():
    """Parameters that are views into a flat buffer, 2 bytes off: the step is
    that of the same weights in storage of their own, bit for bit."""
    torch.manual_seed(3)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=320, num_heads=5, num_kv_heads=5, window=32, num_landmarks_exact=16,
                                        num_landmarks_summary=16).to(DEV, torch.bfloat16).eval()
    st = m.init_state(batch_size=2, device=DEV, dtype=torch.bfloat16)
    x = torch.randn(2, 1, 320, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).bfloat16()
    st2 = state_io.deep_copy_state(st)
    ya, _ = m.step(x, st)
    for lin in (m.q_proj, m.k_proj, m.v_proj, m.lambda_proj, m.write_proj, m.o_proj):
        w = lin.weight
        flat = torch.empty(w.numel() + 1, dtype=w.dtype, device=DEV)
        flat[1:].copy_(w.reshape(-1))
        lin.weight = torch.nn.Parameter(flat[1:].view(w.shape))
        assert lin.weight.data_ptr() % 16
    yb, _ = m.step(x, st2)
    assert torch.equal(ya, yb) and torch.equal(st.k_buf, st2.k_buf) and torch.equal(st.v_buf, st2.v_buf)
