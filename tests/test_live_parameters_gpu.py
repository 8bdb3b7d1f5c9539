"""Calls that read the parameters themselves see every change of one, also
those that torch does not count (through .data, as weights are merged): after
a decode and such a change, the next call is that of a new module that was
given the changed values, bit for bit."""
import copy

import pytest
import torch

import coda_gqa_l
from coda_gqa_l import state_io

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _edit(ts, g):
    for t in ts:
        t.data += 0.3 * torch.randn(t.shape, generator=g, device=DEV).to(t.dtype) * t.float().std(correction=0).clamp_min(0.1).to(t.dtype)


def _values(m):
    return {n: t.detach().clone() for n, t in (*m.named_parameters(), *m.named_buffers())}


def _given(make, values):
    n = make()
    for name, t in (*n.named_parameters(), *n.named_buffers()):
        t.data.copy_(values[name])
    return n


@pytest.mark.parametrize("B,past,L", [(1, 100, 1), (3, 700, 2)])
@torch.no_grad()
def test_unbounded(B, past, L):
    def make():
        return coda_gqa_l.CoDAGQA(embed_dim=512, num_heads=8, num_kv_heads=2).to(DEV, torch.bfloat16).eval()

    torch.manual_seed(1)
    m, g = make(), torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(B, L, 512, generator=g, device=DEV).bfloat16()
    prompt = torch.randn(1, 70, 512, generator=g, device=DEV).bfloat16()
    kv = tuple(torch.randn(B, 2, past, 64, generator=g, device=DEV).bfloat16() for _ in range(2))
    old = m(x, is_causal=False, past_key_value=kv)
    m(prompt)
    for ts in ([m.o_proj.weight], [m.theta], [m.rope.inv_freq], list(m.parameters())):
        _edit(ts, g)
        n = _given(make, _values(m))
        a, b = m(x, is_causal=False, past_key_value=kv), n(x, is_causal=False, past_key_value=kv)
        for s, t in ((a[0], b[0]), (a[1][0], b[1][0]), (a[1][1], b[1][1]), (m(prompt)[0], n(prompt)[0])):
            assert torch.equal(s, t)
        assert not torch.equal(a[0], old[0])
        old = a


@pytest.mark.parametrize("B,dtype,every", [(1, torch.float32, True), (20, torch.float32, True), (70, torch.bfloat16, True),
                                           (2, torch.bfloat16, False)])
@pytest.mark.parametrize("steady", [True, False])
@torch.no_grad()
def test_bounded_step(B, dtype, every, steady):
    def make():
        return coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16, num_landmarks_exact=8,
                                               num_landmarks_summary=8).to(DEV, dtype).eval()

    torch.manual_seed(2)
    m, g = make(), torch.Generator(device=DEV).manual_seed(4)
    st = m.init_state(batch_size=B, device=DEV, dtype=dtype)
    xs = torch.randn(B, 60, 256, generator=g, device=DEV).to(dtype)
    m.prefill_chunked(xs[:, :50 if steady else 7], st, block_size=16, return_outputs=False)
    m.step(xs[:, 50:51], st)
    m.step(xs[:, 51:52], st)
    lins = [m.q_proj, m.k_proj, m.v_proj, m.lambda_proj, m.write_proj, m.o_proj] if every else [m.o_proj]
    for ts in ([p for lin in lins for p in lin.parameters()], [m.rope.inv_freq] if every else []):
        _edit(ts, g)
        n, st2 = _given(make, _values(m)), state_io.deep_copy_state(st)
        x = torch.randn(B, 1, 256, generator=g, device=DEV).to(dtype)
        before = copy.copy(st.pos)
        a, b = m.step(x, st)[0], n.step(x, st2)[0]
        assert torch.equal(a, b) and st.pos == before + 1
        for f in ("k_buf", "v_buf", "g_recent", "allowed", "mem_last_exact"):
            assert torch.equal(getattr(st, f), getattr(st2, f)), f


@pytest.mark.parametrize("B,dtype", [(2, torch.bfloat16), (70, torch.bfloat16), (2, torch.float32)])
@torch.no_grad()
def test_dropped_copies(B, dtype):
    """Every parameter and buffer of a bounded layer changed through .data,
    then drop_parameter_copies()."""
    def make():
        return coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16, num_landmarks_exact=8,
                                               num_landmarks_summary=8).to(DEV, dtype).eval()

    torch.manual_seed(2)
    m, g = make(), torch.Generator(device=DEV).manual_seed(4)
    st = m.init_state(batch_size=B, device=DEV, dtype=dtype)
    xs = torch.randn(B, 60, 256, generator=g, device=DEV).to(dtype)
    m.prefill_chunked(xs[:, :50], st, block_size=16, return_outputs=False)
    m.step(xs[:, 50:51], st)
    m.step(xs[:, 51:52], st)
    _edit([*m.parameters(), *m.buffers()], g)
    m.drop_parameter_copies()
    n, st2 = _given(make, _values(m)), state_io.deep_copy_state(st)
    for part in (xs[:, 52:53], xs[:, 53:54]):
        assert torch.equal(m.step(part, st)[0], n.step(part, st2)[0])
    assert torch.equal(m.prefill_chunked(xs[:, :30], st, block_size=16)[0], n.prefill_chunked(xs[:, :30], st2, block_size=16)[0])
    assert torch.equal(st.k_buf, st2.k_buf) and torch.equal(st.v_buf, st2.v_buf)


@pytest.mark.parametrize("change", ["mul_", "replaced", "data replaced"])
@torch.no_grad()
def test_counted_changes(change):
    """Packed weights and kept RoPE rows (bf16, few rows): changes that torch
    counts need no call."""
    def make():
        return coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16, num_landmarks_exact=8,
                                               num_landmarks_summary=8).to(DEV, torch.bfloat16).eval()

    torch.manual_seed(2)
    m, g = make(), torch.Generator(device=DEV).manual_seed(4)
    st = m.init_state(batch_size=2, device=DEV, dtype=torch.bfloat16)
    xs = torch.randn(2, 60, 256, generator=g, device=DEV).bfloat16()
    m.prefill_chunked(xs[:, :50], st, block_size=16, return_outputs=False)
    for t in range(50, 56, 2):
        m.step(xs[:, t:t + 1], st)
        if change == "mul_":
            m.k_proj.weight.mul_(1.25)
            m.rope.inv_freq.mul_(0.5)
        elif change == "replaced":
            m.k_proj.weight = torch.nn.Parameter(m.k_proj.weight * 1.25)
            m.rope.inv_freq = m.rope.inv_freq * 0.5
        else:
            m.k_proj.weight.data = m.k_proj.weight * 1.25
        n, st2 = _given(make, _values(m)), state_io.deep_copy_state(st)
        assert torch.equal(m.step(xs[:, t + 1:t + 2], st)[0], n.step(xs[:, t + 1:t + 2], st2)[0])
        assert torch.equal(st.k_buf, st2.k_buf)
