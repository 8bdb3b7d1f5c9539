"""The row kernels on a layer's own parameters (coda_project_params,
coda_linear_params, coda_rope_tables): bit for bit what the same kernels give
on packed tiles, at any element address and row stride; tables bit for bit
torch's."""
import pytest
import torch

import coda_gqa_l
from coda_gqa_l import _hip

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _off(w, rows_apart, off):
    """w's values `off` elements past an aligned address, rows farther apart."""
    n, K = w.shape
    flat = torch.full((n * (K + rows_apart) + off,), 9.0, dtype=w.dtype, device=DEV)
    v = flat[off:].view(n, K + rows_apart)[:, :K]
    v.copy_(w)
    return v


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,D,bias,apart,off", [
    (1, 1, 64, False, 0, 0), (3, 17, 64, True, 3, 1), (16, 64, 128, False, 0, 7), (17, 50, 192, True, 8, 0),
    (1, 777, 512, False, 0, 0), (31, 33, 1024, True, 1, 3), (32, 48, 2048, False, 0, 0), (33, 4096, 320, False, 0, 0),
    (64, 100, 2048, True, 5, 2), (65, 63, 1088, False, 0, 0), (128, 6184, 2048, False, 0, 0), (127, 4100, 4096, True, 0, 5),
    (64, 8193, 1024, False, 2, 0), (48, 12300, 1024, True, 0, 0), (20, 8208, 6144, False, 0, 1)])
def test_linear_params_equals_tiles(M, N, D, bias, apart, off, dtype):
    g = torch.Generator(device=DEV).manual_seed(M * 1000 + N)
    w = (torch.randn(N, D, generator=g, device=DEV) * D ** -0.5).to(dtype)
    x = torch.randn(M, D + 8, generator=g, device=DEV).to(dtype)[:, :D]
    b = torch.randn(N, generator=g, device=DEV).to(dtype) if bias else None
    code, st, L = _hip.dtype_code(dtype), _hip.stream_of(x), _hip.lib()
    tiles = torch.empty(-(-N // 64) * 64, D, device=DEV, dtype=dtype)
    _hip.check(L.coda_rows_pack(code, w.data_ptr(), N, D, D, tiles.data_ptr(), st))
    ld = N + (-N) % 4 + 4
    want, got = (torch.full((M + 1, ld), 7.0, device=DEV, dtype=dtype) for _ in range(2))
    bf = b.float() if bias else None
    _hip.check(L.coda_linear_rows(code, x.data_ptr(), x.stride(0), M, tiles.data_ptr(), N, D, _hip.ptr(bf),
                                  want.data_ptr(), ld, st))
    v = _off(w, apart, off)
    _hip.check(L.coda_linear_params(code, x.data_ptr(), x.stride(0), M, v.data_ptr(), v.stride(0), N, D, _hip.ptr(b),
                                    got.data_ptr(), ld, st))
    assert torch.equal(got, want)


@pytest.mark.parametrize("B,D,H,Hkv,inter,gate,dtype", [
    (1, 512, 8, 2, True, True, "bf16"), (3, 320, 5, 5, False, True, "f32"), (17, 4096, 32, 8, False, False, "bf16"),
    (33, 256, 4, 2, False, True, "bf16"), (64, 1024, 16, 4, True, True, "bf16"), (100, 2048, 16, 2, False, True, "bf16"),
    (32, 1024, 8, 1, True, False, "f32"), (128, 192, 3, 1, True, True, "bf16"), (1, 64, 1, 1, False, True, "bf16"),
    (2, 128, 4, 2, False, True, "f32")])
@pytest.mark.parametrize("inv", [torch.float32, torch.bfloat16])
@torch.no_grad()
def test_project_params_equals_packed(B, D, H, Hkv, inter, gate, dtype, inv):
    dt = torch.float32 if dtype == "f32" else torch.bfloat16
    torch.manual_seed(B + D)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(
        embed_dim=D, num_heads=H, num_kv_heads=Hkv, window=16, num_landmarks_exact=8, num_landmarks_summary=8,
        rope_interleaved=inter, **({} if gate else {"write_policy": "none"})).to(DEV, dt).eval()
    Dh, g = D // H, torch.Generator(device=DEV).manual_seed(2)
    rows = [m.q_proj, m.k_proj, m.v_proj, m.lambda_proj] + ([m.write_proj] if gate else [])
    for i, lin in enumerate(rows):
        lin.bias = torch.nn.Parameter(torch.randn(lin.out_features, generator=g, device=DEV).to(dt)) if i != 2 else None
        lin.weight = torch.nn.Parameter(_off(lin.weight, 0, i) if i % 2 else lin.weight)
    m.rope.inv_freq = m.rope.inv_freq.to(inv)
    m.theta.copy_(m.theta + torch.randn(m.theta.shape, generator=g, device=DEV))
    x, p0 = torch.randn(B, 1, D, generator=g, device=DEV).to(dt), 5003
    cos, sin = (t.contiguous() for t in m.rope(seq_len=1, offset=p0, device=torch.device("cuda:0"), dtype=dt))
    lib, st, outs = _hip.lib(), _hip.stream_of(x), []
    tabs = [torch.zeros((n, Dh // 2), dtype=dt, device=DEV) for n in (1, 1, H, H)]
    for packed in (True, False):
        d = m._proj_desc(x, B, 1, cos, sin)
        o = [torch.full((B, n), 7.0, dtype=dt, device=DEV) for n in (D, Hkv * Dh, Hkv * Dh, H)]
        gt = torch.full((B,), 7.0, device=DEV)
        d.x, d.x_sm = x.data_ptr(), D
        d.q, d.q_sm, d.k, d.k_sm, d.v, d.v_sm = o[0].data_ptr(), D, o[1].data_ptr(), Hkv * Dh, o[2].data_ptr(), Hkv * Dh
        d.lam, d.lam_sm, d.g = o[3].data_ptr(), H, gt.data_ptr()
        if packed:
            w, b, d.w_layout = m._proj_pack(dt)
            d.w, d.bias = w.data_ptr(), b.data_ptr()
            _hip.check(lib.coda_project_rows(d, st))
        else:
            p = m._proj_params(m._plain_rows(x, "q_proj", "k_proj", "v_proj", "lambda_proj",
                                             *(("write_proj",) if gate else ())))
            d.rope_cos = d.rope_sin = None
            p.inv_freq, p.inv_dtype, p.p0 = m.rope.inv_freq.data_ptr(), _hip.dtype_code(inv), p0
            p.theta, p.theta_dtype = m.theta.data_ptr(), _hip.dtype_code(dt)
            p.rope_cos, p.rope_sin, p.theta_cos, p.theta_sin = (t.data_ptr() for t in tabs)
            _hip.check(lib.coda_project_params(d, p, st))
        outs.append(o + [gt])
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    assert torch.equal(tabs[0], cos) and torch.equal(tabs[1], sin)
    assert torch.equal(tabs[2], torch.cos(m.theta)) and torch.equal(tabs[3], torch.sin(m.theta))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("inv", [torch.bfloat16, torch.float32])
@torch.no_grad()
def test_tables_equal_the_module(dtype, inv):
    m = coda_gqa_l.CoDAGQA(embed_dim=256, num_heads=2, num_kv_heads=1).to(DEV).eval()
    m.rope.inv_freq = m.rope.inv_freq.to(inv)
    dev = torch.device("cuda:0")
    for p0, L in ((0, 1), (0, 65536), (4095, 3), (1 << 20, 777), ((1 << 24) - 9, 9), ((1 << 24) - 8, 9)):
        for got, want in zip(m._rope_tables(p0, L, dev, dtype), m.rope(seq_len=L, offset=p0, device=dev, dtype=dtype)):
            assert got.shape == want.shape and got.is_contiguous() and torch.equal(got, want), (p0, L)


@pytest.mark.parametrize("B,D,H,Hkv,inter,gate", [(1, 512, 8, 2, True, True), (9, 320, 5, 5, False, True),
                                                  (33, 256, 4, 2, False, False), (2, 4096, 32, 8, False, True)])
@pytest.mark.parametrize("half_bias", [False, True])
@torch.no_grad()
def test_pack_in_one_launch(B, D, H, Hkv, inter, gate, half_bias):
    """The packed form from the parameters, any address, against the one from
    a concatenation (taken where a dtype differs: here fp32 copies of the same
    values)."""
    torch.manual_seed(D)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(
        embed_dim=D, num_heads=H, num_kv_heads=Hkv, window=16, num_landmarks_exact=8, num_landmarks_summary=8,
        rope_interleaved=inter, **({} if gate else {"write_policy": "none"})).to(DEV, torch.bfloat16).eval()
    lins = [m.q_proj, m.k_proj, m.v_proj, m.lambda_proj] + ([m.write_proj] if gate else [])
    for i, lin in enumerate(lins):
        lin.weight = torch.nn.Parameter(_off(lin.weight, i, i))
        lin.bias = torch.nn.Parameter(torch.randn(lin.out_features, device=DEV).bfloat16()) if (i % 2) != half_bias else None
    w, b, layout = m._proj_pack(torch.bfloat16)
    for lin in lins:
        lin.float()
    m.drop_parameter_copies()
    w2, b2, layout2 = m._proj_pack(torch.bfloat16)
    assert layout == layout2 == 1 and torch.equal(w, w2) and torch.equal(b, b2)
