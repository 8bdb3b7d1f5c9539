"""Decode calls in captured graphs: the first call of a layer may be the
captured one, later eager calls leave what the graph reads alone, and a graph
whose parameters change reads the changed values."""
import pytest
import torch

import coda_gqa_l
from coda_gqa_l import state_io

pytestmark = pytest.mark.gpu
DEV = "cuda"
FIELDS = ("k_buf", "v_buf", "allowed", "g_recent", "mem_last_exact", "_exact_v_norm", "_sum_lf_k_norm")


def _capture(fn):
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            out = fn()
    torch.cuda.current_stream().wait_stream(side)
    return graph, out


@pytest.mark.parametrize("first", [True, False])
@torch.no_grad()
def test_unbounded_decode(first):
    def make():
        torch.manual_seed(1)
        return coda_gqa_l.CoDAGQA(embed_dim=512, num_heads=8, num_kv_heads=2).to(DEV, torch.bfloat16).eval()

    m, plain = make(), make()
    g = torch.Generator(device=DEV).manual_seed(2)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()  # noqa: E731
    x, kv, long = rnd(2, 1, 512), (rnd(2, 2, 100, 64), rnd(2, 2, 100, 64)), (rnd(2, 2, 9000, 64), rnd(2, 2, 9000, 64))
    run = lambda m, kv: m(x, is_causal=False, past_key_value=kv)  # noqa: E731
    want, want_long = run(plain, kv), run(plain, long)[0]
    torch.cuda.synchronize()
    if not first:
        run(m, kv)
    graph, (y, (k, v)) = _capture(lambda: run(m, kv))
    # before any replay: an eager call of the layer
    assert torch.equal(run(m, kv)[0], want[0])
    for rep in range(3):
        for t in (y, k, v):
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in ((y, want[0]), (k, want[1][0]), (v, want[1][1])):
            assert torch.equal(a, b), f"replay {rep}"
        # a longer past, a long prompt, and tensors that take any freed memory
        assert torch.equal(run(m, long)[0], want_long)
        m(rnd(1, 5000, 512))
        junk = [torch.full((1 << n,), float("nan"), device=DEV) for n in range(8, 22)]
        del junk
    m.o_proj.weight.mul_(0.5)
    plain.o_proj.weight.mul_(0.5)
    run(m, kv)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, run(plain, kv)[0])


@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("B,dtype", [(2, torch.bfloat16), (70, torch.bfloat16), (2, torch.float32)])
@torch.no_grad()
def test_bounded_projections(B, dtype, first):
    """The step's projections (the part of a step that reads weights and
    tables): captured as a layer's first call or a later one."""
    def make():
        torch.manual_seed(1)
        return coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16,
                                               num_landmarks_exact=8, num_landmarks_summary=8).to(DEV, dtype).eval()

    m, plain = make(), make()
    g = torch.Generator(device=DEV).manual_seed(2)
    x = torch.randn(B, 1, 256, generator=g, device=DEV).to(dtype)
    want = [t.clone() for t in plain._front(x, 77, fused=True)]
    y_want = plain._out_rows(x).clone()
    torch.cuda.synchronize()
    if not first:
        m._front(x, 77, fused=True)
    graph, out = _capture(lambda: (*m._front(x, 77, fused=True), m._out_rows(x)))
    for a, b in zip(m._front(x, 77, fused=True), want):  # eager, before any replay
        assert torch.equal(a, b)
    for rep in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want + [y_want]):
            assert torch.equal(a, b), f"replay {rep}"
        m._front(x, 9000, fused=True)  # (past any table kept so far)
        junk = [torch.full((1 << n,), float("nan"), device=DEV) for n in range(8, 22)]
        del junk


@pytest.mark.parametrize("warm", [1, 3])
@pytest.mark.parametrize("B,dtype", [(2, torch.bfloat16), (70, torch.bfloat16), (2, torch.float32)])
@torch.no_grad()
def test_bounded_step(B, dtype, warm):
    """A whole steady-state step, captured after eager ones (the landmark
    rates are made on the host once)."""
    def make():
        torch.manual_seed(1)
        return coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=256, num_heads=4, num_kv_heads=2, window=16,
                                               num_landmarks_exact=8, num_landmarks_summary=8).to(DEV, dtype).eval()

    m = make()
    g = torch.Generator(device=DEV).manual_seed(2)
    x = torch.randn(B, 60, 256, generator=g, device=DEV).to(dtype)
    st = m.init_state(batch_size=B, device=DEV, dtype=dtype)
    m.prefill_chunked(x[:, :40], st, block_size=16, return_outputs=False)
    for t in range(warm):
        m.step(x[:, 40 + t:41 + t], st)
    st = state_io.deep_copy_state(st)
    start, other = {f: getattr(st, f).clone() for f in FIELDS}, state_io.deep_copy_state(st)
    xt = x[:, 50:51].contiguous()
    want = make().step(xt, other)[0].clone()
    torch.cuda.synchronize()
    graph, y = _capture(lambda: m.step(xt, st)[0])
    for rep in range(3):
        for f in FIELDS:
            getattr(st, f).copy_(start[f])
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), f"replay {rep}"
        for f in FIELDS:
            assert torch.equal(getattr(st, f), getattr(other, f)), f
        # eager steps of another state through the same layer
        st3 = state_io.deep_copy_state(other)
        st3.pos = 9000
        for _ in range(2):
            m.step(xt, st3)
