"""The work that users of coda_gqa_l have it do, as cases to time and compare.

Kinds of case, each one call of a public entry point:

  step       CoDAGQALandmarkPerf2.step: one decode token of a bounded layer
             (projections, bank update, attention, output projection) in the
             steady state: full ring, filled banks
  prefill    CoDAGQALandmarkPerf2.prefill_chunked: a prompt or the next part
             of a stream, in chunks; through EveCoDAAdapter / LlamaCoDAAdapter
             for the models that hold one
  attn       diff_flash_attn, the attention operator alone, causal
  unbounded  CoDAGQA.forward, the layer without a bound: a whole prompt, or a
             decode token on top of its K/V

Values: activations N(0, 1), weights as nn.Linear draws them with the query
projection scaled so that attention scores have a spread of about 1, write
gates on both sides of their thresholds, a lambda that matters.  Bank
decisions follow from these as in a trained layer: most evicted tokens are
novel, some are gated out.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "coda-gqa-l_amd"))
import coda_gqa_l  # noqa: E402
from coda_gqa_l import state_io  # noqa: E402
from coda_gqa_l.state import CoDAGQALandmarkStatePerf2  # noqa: E402

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
TOKENS = 32  # distinct decode inputs of a state, taken in turn


def _layer(kind, D, H, Hkv, B, dtype="bf16", **more):
    return dict(kind=kind, D=D, H=H, Hkv=Hkv, B=B, dtype=dtype, **more)


_MEDIUM = dict(W=256, Me=64, Ms=64)
_LARGE = dict(W=512, Me=128, Ms=128)


def listed():
    return [
        # one user's chat on the 7B-shaped layer: latency of a token
        dict(name="step_7b_b1", **_layer("step", 4096, 32, 8, 1, **_MEDIUM)),
        # a serving batch on the same layer
        dict(name="step_7b_b64", **_layer("step", 4096, 32, 8, 64, **_MEDIUM)),
        # a large serving batch on the 70B-shaped layer, large cache
        dict(name="step_70b_b128", **_layer("step", 8192, 64, 8, 128, **_LARGE)),
        # the small fp32 model (research, tests): launches and host work
        dict(name="step_512_f32", **_layer("step", 512, 8, 2, 1, "f32", **_MEDIUM)),
        # its prompt of 2048 tokens from an empty cache
        dict(name="prefill_512_f32", **_layer("prefill", 512, 8, 2, 1, "f32", L=2048, block=256, fresh=True,
                                               adapter="", **_MEDIUM)),
        # one user's prompt, of no round length, from an empty cache
        dict(name="prefill_7b_prompt", **_layer("prefill", 4096, 32, 8, 1, L=1999, block=256, fresh=True, adapter="",
                                                 **_MEDIUM)),
        # four long documents streamed in parts of 8192 tokens
        dict(name="prefill_7b_stream", **_layer("prefill", 4096, 32, 8, 4, L=8192, block=256, fresh=False,
                                                 adapter="", **_MEDIUM)),
        # eight streams through the 70B-shaped layer
        dict(name="prefill_70b_stream", **_layer("prefill", 8192, 64, 8, 8, L=2048, block=256, fresh=False,
                                                  adapter="", **_LARGE)),
        # two prompts through a multi-head model with head_dim 64 and its adapter's block of 1024
        dict(name="prefill_eve_prompt", **_layer("prefill", 1024, 16, 16, 2, L=1500, block=1024, fresh=True,
                                                  adapter="eve", **_MEDIUM)),
        # causal attention of the unbounded layer at full length
        dict(name="attn_causal_8k", kind="attn", dtype="bf16", B=2, H=32, Hkv=8, Dh=128, Lq=8192, Lk=8192),
        # a small model's odd-sized chunk on top of a longer context
        dict(name="attn_ragged_512", kind="attn", dtype="bf16", B=1, H=8, Hkv=2, Dh=64, Lq=777, Lk=4097),
        # decode of the unbounded layer on top of 4096 tokens
        dict(name="unbounded_decode_7b", **_layer("unbounded", 4096, 32, 8, 4, Lq=1, past=4096)),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng, most):
    """(D, H, Hkv): head_dim 64 or 128, 1 to 8 query heads per KV head."""
    while True:
        Dh, G, Hkv = rng.choice((64, 128)), rng.choice((1, 2, 4, 4, 8)), rng.choice((1, 2, 4, 8, 8, 16))
        if 256 <= Dh * G * Hkv <= most:
            return Dh * G * Hkv, G * Hkv, Hkv


def draw(rng):
    kind = rng.choice(("step", "step", "prefill", "prefill", "attn", "unbounded"))
    f32 = rng.random() < 0.2
    dtype = "f32" if f32 else "bf16"
    if kind == "attn":
        Dh, G, Hkv = rng.choice((64, 128)), rng.choice((1, 2, 4, 8)), rng.choice((1, 2, 4, 8))
        B, Lq = rng.choice((1, 1, 2, 3)), _log(rng, 64, 1024 if f32 else 4096)
        Lk = Lq if rng.random() < 0.5 else min(8192, Lq + _log(rng, 1, 1024 if f32 else 4096))
        return dict(kind=kind, dtype=dtype, B=B, H=G * Hkv, Hkv=Hkv, Dh=Dh, Lq=Lq, Lk=Lk)
    if kind == "unbounded":
        D, H, Hkv = _heads(rng, 1024 if f32 else 4096)
        B = _log(rng, 1, 8)
        if rng.random() < 0.6:
            return _layer(kind, D, H, Hkv, B, dtype, Lq=1, past=_log(rng, 100, 8191))
        return _layer(kind, D, H, Hkv, min(B, 2), dtype, Lq=_log(rng, 32, 1024 if f32 else 4096), past=0)
    W = rng.choice((128, 256, 256, 512, _log(rng, 64, 512)))
    Me, Ms = rng.choice(((64, 64), (64, 64), (32, 32), (128, 128), (_log(rng, 16, 128), _log(rng, 16, 128))))
    D, H, Hkv = _heads(rng, 1024 if f32 else 8192 if kind == "step" else 4096)
    if kind == "step":
        return _layer(kind, D, H, Hkv, _log(rng, 1, 16 if f32 else 128), dtype, W=W, Me=Me, Ms=Ms)
    B, L = _log(rng, 1, 8), _log(rng, 200, 2048 if f32 else 8192)
    while B > 1 and B * L * D > 4 * 8192 * (512 if f32 else 4096):
        B -= 1
    if rng.random() < 0.2:  # window only
        Me = Ms = 0
    adapter = "eve" if H == Hkv and rng.random() < 0.7 else "llama" if rng.random() < 0.3 else ""
    return _layer(kind, D, H, Hkv, B if not f32 else min(B, 2), dtype, L=L, block=rng.choice((128, 256, 256, 512, 1024)),
                  fresh=rng.random() < 0.5, adapter=adapter, W=W, Me=Me, Ms=Ms)


# ----------------------------------------------------------------- prepare
def _randn(gen, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(*shape, generator=gen, device=DEV) * std).to(dtype)


def _settle(m, gen):
    """Weights as a trained layer has them in the respects that steer the
    path: score spread, write gates, lambda, noise angles, norm weights."""
    D = m.embed_dim
    with torch.no_grad():
        for lin in (m.q_proj, m.k_proj, m.v_proj, m.o_proj, m.lambda_proj):
            lin.weight.uniform_(-D ** -0.5, D ** -0.5, generator=gen)
        m.q_proj.weight.mul_(3.0)
        m.lambda_proj.bias.copy_(_randn(gen, m.num_heads, std=0.5) - 1.0)
        m.theta.copy_(m.theta + _randn(gen, *m.theta.shape, std=0.1))
        if m.head_norm_mode == "full":
            m.head_norm.weight.copy_(1.0 + _randn(gen, m.head_dim, std=0.1))
        if hasattr(m, "write_proj"):
            m.write_proj.weight.copy_(_randn(gen, 1, D, std=0.7 * D ** -0.5))
            m.write_proj.bias.fill_(-2.0)
            m.summary_eta_logit.copy_(-3.0 + _randn(gen, m.num_kv_heads, std=0.5))


def _bounded(c, gen):
    """(callable module, its bounded layer)."""
    dt = DTYPES[c["dtype"]]
    sizes = dict(window=c["W"], num_landmarks_exact=c["Me"], num_landmarks_summary=c["Ms"])
    with torch.device(DEV):
        if c.get("adapter") == "eve":
            host = coda_gqa_l.EveCoDAAdapter(c["D"], c["H"], c["D"] // c["H"], bounded=True, block_size=c["block"],
                                             **sizes)
        elif c.get("adapter") == "llama":
            host = coda_gqa_l.LlamaCoDAAdapter(c["D"], c["H"], c["Hkv"], c["D"] // c["H"], bounded=True,
                                               block_size=c["block"], **sizes)
        else:
            host = coda_gqa_l.CoDAGQALandmarkPerf2(embed_dim=c["D"], num_heads=c["H"], num_kv_heads=c["Hkv"], **sizes)
    m = host.coda if c.get("adapter") else host
    _settle(m, gen)
    if c.get("adapter") == "eve":  # its projections carry biases
        D, bias = c["D"], lambda n: _randn(gen, n, std=0.02)  # noqa: E731
        host.load_eve_weights(c_attn_weight=torch.cat([m.q_proj.weight, m.k_proj.weight, m.v_proj.weight]).detach(),
                              c_attn_bias=bias(3 * D), c_proj_weight=m.o_proj.weight.detach(), c_proj_bias=bias(D))
    host = host.to(device=DEV, dtype=dt).eval()
    return host, m


def _unit(x):
    return F.normalize(x.float(), dim=-1, eps=1e-6)


def _steady_state(c, gen, pos=4096):
    """A layer's cache after a few thousand tokens: full ring, filled banks."""
    dt, B, Hkv, Dh, W, Me, Ms = DTYPES[c["dtype"]], c["B"], c["Hkv"], c["D"] // c["H"], c["W"], c["Me"], c["Ms"]
    k = _randn(gen, B, Hkv, W + Me + Ms, Dh, std=3 ** -0.5)
    v = _randn(gen, B, Hkv, W + Me + Ms, Dh, std=3 ** -0.5)
    # prototypes: the low-frequency band alone, both averaged down
    k[:, :, W + Me:, :Dh // 2] = 0
    k[:, :, W + Me:] *= 0.7
    v[:, :, W + Me:] *= 0.5
    k, v = k.to(dt), v.to(dt)
    age = torch.stack([torch.randperm(pos - W, generator=gen, device=DEV)[:Me] for _ in range(B)])
    return CoDAGQALandmarkStatePerf2(
        k_buf=k, v_buf=v, allowed=torch.ones((B, W + Me + Ms), dtype=torch.bool, device=DEV),
        g_recent=torch.sigmoid(_randn(gen, B, W, std=0.7) - 2.0).to(dt).float(), recent_idx=0, recent_filled=W,
        mem_last_exact=age.reshape(B, Me).to(torch.int64), pos=pos, active_exact=Me, active_summary=Ms,
        _exact_v_norm=_unit(v[:, :, W:W + Me]).to(dt).contiguous() if Me else None,
        _sum_lf_k_norm=_unit(k[:, :, W + Me:, Dh // 2:]).to(dt).contiguous() if Ms else None)


def prepare(case, seed):
    c, gen = case, torch.Generator(device=DEV).manual_seed(seed)
    dt = DTYPES[c["dtype"]]
    if c["kind"] == "attn":
        B, H, Hkv, Dh, Lq, Lk = c["B"], c["H"], c["Hkv"], c["Dh"], c["Lq"], c["Lk"]
        q = _randn(gen, B, H, Lq, Dh, dtype=dt)
        r = torch.linalg.qr(_randn(gen, H, Dh, Dh))[0]  # the noise rotation of each head
        return dict(c=c, q=q, q_noise=(q.float() @ r).to(dt), k=_randn(gen, B, Hkv, Lk, Dh, dtype=dt),
                    v=_randn(gen, B, Hkv, Lk, Dh, dtype=dt),
                    lam=(0.1 + 0.8 * torch.rand(B, H, Lq, 1, generator=gen, device=DEV)).to(dt),
                    w=(1.0 + _randn(gen, Dh, std=0.1)).to(dt))
    if c["kind"] == "unbounded":
        with torch.device(DEV):
            m = coda_gqa_l.CoDAGQA(embed_dim=c["D"], num_heads=c["H"], num_kv_heads=c["Hkv"])
        _settle(m, gen)
        m = m.to(device=DEV, dtype=dt).eval()
        past = None
        if c["past"]:
            past = tuple(_randn(gen, c["B"], c["Hkv"], c["past"], m.head_dim, dtype=dt, std=3 ** -0.5)
                         for _ in range(2))
        return dict(c=c, m=m, x=_randn(gen, c["B"], c["Lq"], c["D"], dtype=dt), past=past)
    host, m = _bounded(c, gen)
    if c["kind"] == "step":
        return dict(c=c, m=m, st=_steady_state(c, gen), i=0,
                    xs=[_randn(gen, c["B"], 1, c["D"], dtype=dt) for _ in range(TOKENS)])
    if c["fresh"]:
        torch.manual_seed(seed)  # init_state draws its landmarks from the CPU generator
        st = m.init_state(batch_size=c["B"], device=DEV, dtype=dt)
    else:
        st = _steady_state(c, gen)
    return dict(c=c, host=host, m=m, st=st, x=_randn(gen, c["B"], c["L"], c["D"], dtype=dt))


# --------------------------------------------------------------------- run
def _with_state(y, st):
    return dict(y=y, k=st.k_buf, v=st.v_buf, allowed=st.allowed, gates=st.g_recent, last=st.mem_last_exact,
                exact_norm=st._exact_v_norm, summary_norm=st._sum_lf_k_norm)


def run(s):
    c = s["c"]
    with torch.no_grad():
        if c["kind"] == "attn":
            return coda_gqa_l.diff_flash_attn(s["q"], s["q_noise"], s["k"], s["v"], s["lam"], s["w"], is_causal=True)
        if c["kind"] == "unbounded":
            y, (k, v) = s["m"](s["x"], is_causal=s["past"] is None, past_key_value=s["past"])
            return dict(y=y, k=k, v=v)
        if c["kind"] == "step":
            x = s["xs"][s["i"] % TOKENS]
            s["i"] += 1
            y, s["st"] = s["m"].step(x, s["st"])
            return _with_state(y, s["st"])
        # a prompt starts from a copy of the empty cache; a stream goes on
        st = state_io.deep_copy_state(s["st"]) if c["fresh"] else s["st"]
        if c["adapter"]:
            s["host"].set_state(st)
            y = s["host"](s["x"])
            y, st = y[0] if isinstance(y, tuple) else y, s["host"].get_state()
        else:
            y, st = s["m"].prefill_chunked(s["x"], st, block_size=c["block"])
        if not c["fresh"]:
            s["st"] = st
        return _with_state(y, st)


# -------------------------------------------------------------------- work
def work(case):
    c = case
    e = 2 if c["dtype"] == "bf16" else 4
    B, H, Hkv = c["B"], c["H"], c["Hkv"]
    if c["kind"] == "attn":
        Lq, Lk, Dh = c["Lq"], c["Lk"], c["Dh"]
        return dict(bytes=e * (3 * B * H * Lq * Dh + 2 * B * Hkv * Lk * Dh + B * H * Lq),
                    flops=8 * Dh * B * H * (Lq * (Lk - Lq) + Lq * (Lq + 1) / 2))
    D, Dh = c["D"], c["D"] // c["H"]
    feats = 2 * D + 2 * Hkv * Dh + H + (0 if c["kind"] == "unbounded" else 1)
    L = c.get("Lq", 1) if c["kind"] != "prefill" else c["L"]
    weights, gemm = feats * D * e, 2.0 * feats * D * B * L
    io = 2 * B * L * D * e
    if c["kind"] == "unbounded":
        Lk = c["past"] + L
        pairs = L * c["past"] + (L * (L + 1) / 2 if L > 1 else 1)
        return dict(bytes=weights + io + 2 * B * Hkv * Dh * e * (c["past"] + Lk), flops=gemm + 8 * Dh * B * H * pairs)
    W, bank = c["W"], c["Me"] + c["Ms"]
    state = B * (2 * Hkv * (W + bank) * Dh * e + Hkv * (c["Me"] * Dh + c["Ms"] * Dh // 2) * e + 4 * W + W + bank + 8 * c["Me"])
    if c["kind"] == "step":
        # the cache is read once; a ring slot, an exact and a summary slot are rewritten
        return dict(bytes=weights + io + state + 6 * B * Hkv * Dh * e, flops=gemm + 8 * Dh * B * H * (W + bank))
    pairs = 0
    for t in range(0, L, c["block"]):
        n = min(c["block"], L - t)
        seen = W + bank if not c["fresh"] else min(W + bank, t)
        pairs += n * seen + n * (n + 1) / 2
    return dict(bytes=weights + io + 2 * state, flops=gemm + 8 * Dh * B * H * pairs)


def tolerance(case):
    # about four times the distance from exact() that was measured: 5.8e-7 in
    # fp32, 2.7e-3 for the bf16 attention operator, 5.6e-3 for bf16 layers
    if case["dtype"] == "f32":
        return {"rel": 5e-6, "max": 1e-4}
    return {"rel": 1e-2, "max": 0.1} if case["kind"] == "attn" else {"rel": 2e-2, "max": 0.2}


# ------------------------------------------------------- the same in 64 bits
def _rotate(x, cos, sin, interleaved=True):
    if interleaved:
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], dim=-1).flatten(-2)
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _angles(m, p0, L):
    """The layer's RoPE angles: positions and products in the buffer's type."""
    inv = m.rope.inv_freq
    t = torch.arange(p0, p0 + L, device=DEV, dtype=inv.dtype)
    return (t[:, None] * inv[None, :]).double()


def _linear(lin, x):
    y = x @ lin.weight.double().t()
    return y if lin.bias is None else y + lin.bias.double()


def _norm(y, w, eps):
    return y if w is None else y * torch.rsqrt(y.square().mean(-1, keepdim=True) + eps) * w.double()


def _attend(q, qn, k, v, lam, w, eps, visible):
    """q, qn (B,H,Lq,Dh), k, v (B,Hkv,Lk,Dh), lam (B,H,Lq,1); visible (Lq, Lk) or None."""
    B, H, Lq, Dh = q.shape
    G, out = H // k.shape[1], torch.empty_like(q)
    for b in range(B):
        for h in range(H):
            kk, vv = k[b, h // G], v[b, h // G]
            for t in range(0, Lq, 1024):
                y = []
                for x in (q, qn):
                    sc = x[b, h, t:t + 1024] @ kk.t() / math.sqrt(Dh)
                    if visible is not None:
                        sc = sc.masked_fill(~visible[t:t + 1024], -math.inf)
                    y.append(torch.softmax(sc, dim=-1) @ vv)
                out[b, h, t:t + 1024] = _norm(y[0] - lam[b, h, t:t + 1024] * y[1], w, eps)
    return out


def _project(m, x, p0, interleaved):
    B, L, _ = x.shape
    x, a = x.double(), _angles(m, p0, L)
    heads = lambda y, n: y.view(B, L, n, m.head_dim).transpose(1, 2)  # noqa: E731
    q = _rotate(heads(_linear(m.q_proj, x), m.num_heads), a.cos(), a.sin(), interleaved)
    k = _rotate(heads(_linear(m.k_proj, x), m.num_kv_heads), a.cos(), a.sin(), interleaved)
    th = m.theta.double()[:, None]
    qn = _rotate(q, th.cos(), th.sin())
    lam = torch.sigmoid(_linear(m.lambda_proj, x)).transpose(1, 2).unsqueeze(-1)
    return q, qn, k, heads(_linear(m.v_proj, x), m.num_kv_heads), lam


def _out(m, heads):
    B, H, L, Dh = heads.shape
    return _linear(m.o_proj, heads.transpose(1, 2).reshape(B, L, H * Dh))


def _weight(m):
    return m.head_norm.weight if m.head_norm_mode == "full" else None


def _write_token(m, st, k_new, v_new, g_new):
    """One token into the cache in 64 bits: the evicted token updates the
    exact bank (novel tokens take the least recently used slot) and the
    summary bank (the nearest prototype moves towards it)."""
    W, Me, Ms, lf = m.window, m.Me, m.Ms, m.lf_start
    B, rows = k_new.shape[0], torch.arange(k_new.shape[0], device=DEV)
    j = st.recent_idx
    k, v, allowed, gates = st.k_buf.double(), st.v_buf.double(), st.allowed.clone(), st.g_recent.clone()
    last = st.mem_last_exact.clone()
    en = None if st._exact_v_norm is None else st._exact_v_norm.double()
    sn = None if st._sum_lf_k_norm is None else st._sum_lf_k_norm.double()
    ke, ve, g = k[:, :, j].clone(), v[:, :, j].clone(), gates[:, j]
    unit = lambda x: F.normalize(x, dim=-1, eps=1e-6)  # noqa: E731
    if Me:
        best, at = torch.einsum("bhd,bhmd->bhm", unit(ve), en).mean(1).max(-1)
        novel, keep = best < m.exact_novelty_threshold, g >= m.write_gate_threshold_exact
        idx = torch.where(novel, last.argmin(-1), at)
        write = novel | (best >= m.exact_match_threshold) if m.exact_refresh_on_hit else novel
        for b in rows[write & keep].tolist():
            k[b, :, W + idx[b]], v[b, :, W + idx[b]], en[b, :, idx[b]] = ke[b], ve[b], unit(ve[b])
        last[rows[keep], idx[keep]] = st.pos - W
    if Ms:
        idx = torch.einsum("bhd,bhmd->bhm", unit(ke[..., lf:]), sn).mean(1).argmax(-1)
        keep = g >= m.write_gate_threshold_summary
        eta = torch.sigmoid(m.summary_eta_logit.double())[None, :, None] * g.double()[:, None, None]
        for b in rows[keep].tolist():
            i = W + Me + idx[b]
            k[b, :, i, lf:] += eta[b] * (ke[b, :, lf:] * m.energy_scale - k[b, :, i, lf:])
            v[b, :, i] += eta[b] * (ve[b] - v[b, :, i])
            sn[b, :, idx[b]] = unit(k[b, :, i, lf:])
    k[:, :, j], v[:, :, j], gates[:, j] = k_new, v_new, g_new.float()
    return dict(k=k, v=v, allowed=allowed, gates=gates.double(), last=last, exact_norm=en, summary_norm=sn)


def exact(case, seed):
    c, s = case, prepare(case, seed)
    with torch.no_grad():
        if c["kind"] == "attn":
            Lq, Lk = c["Lq"], c["Lk"]
            vis = torch.arange(Lk, device=DEV)[None] <= torch.arange(Lk - Lq, Lk, device=DEV)[:, None]
            return _attend(*(s[n].double() for n in ("q", "q_noise", "k", "v", "lam")), s["w"], 1e-6, vis)
        m = s["m"]
        if c["kind"] == "unbounded":
            q, qn, k, v, lam = _project(m, s["x"], c["past"], True)
            if s["past"] is not None:
                k, v = (torch.cat([p.double(), x], 2) for p, x in zip(s["past"], (k, v)))
            L = c["Lq"]
            vis = None if c["past"] else torch.ones(L, L, dtype=torch.bool, device=DEV).tril()
            return dict(y=_out(m, _attend(q, qn, k, v, lam, _weight(m), m._eps, vis)), k=k, v=v)
        st, x = s["st"], s["xs"][0] if c["kind"] == "step" else s["x"]
        q, qn, k, v, lam = _project(m, x, st.pos, m.rope_interleaved)
        g = torch.sigmoid(_linear(m.write_proj, x.double())).squeeze(-1)
        if c["kind"] == "step":
            r = _write_token(m, st, k[:, :, 0], v[:, :, 0], g[:, 0])
            return dict(r, y=_out(m, _attend(q, qn, r["k"], r["v"], lam, _weight(m), m._eps, None)))
        if c["Me"] + c["Ms"] > 0:
            # candidates are ranked by rounded gates, ties in the order of a
            # partial sort: slots have no counterpart in 64 bits
            return None
        W, L = c["W"], c["L"]
        n0 = st.recent_filled
        kk, vv = torch.cat([st.k_buf[:, :, :n0].double(), k], 2), torch.cat([st.v_buf[:, :, :n0].double(), v], 2)
        i, t = torch.arange(n0 + L, device=DEV)[None], torch.arange(L, device=DEV)[:, None]
        start = n0 + t // c["block"] * c["block"]
        y = _out(m, _attend(q, qn, kk, vv, lam, _weight(m), m._eps, (i <= n0 + t) & (i >= start - W)))
        full = n0 + L >= W
        return dict(y=y, k=kk[:, :, -W:] if full else None, v=vv[:, :, -W:] if full else None, allowed=None, gates=None,
                    last=None, exact_norm=None, summary_norm=None)
