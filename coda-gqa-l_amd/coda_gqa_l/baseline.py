"""Unbounded differential attention (the Phase-1 layer), on MI355X.

Same constructor, parameters and forward contract as the reference's
CoDAGQA (src/coda_gqa_l/baseline.py:22-147): returns (y, (k_total,
v_total)).  RoPE of keys runs in the rope kernel; RoPE of queries, the noise
rotation, GQA sharing, the causal mask, the lambda difference and the head
norm run inside one attention kernel (no repeat_kv copies, one K/V pass).
"""

from __future__ import annotations

import ctypes
import math
from typing import Optional, Tuple

import torch
import torch.nn as nn

from . import _hip, ops
from .primitives import HeadwiseRMSNorm, RotaryEmbedding, apply_rope
from .rows import RowsMixin, _aligned


class CoDAGQA(RowsMixin, nn.Module):
    def __init__(self, *, embed_dim: int, num_heads: int, num_kv_heads: int, rope_base: float = 10_000.0,
                 lambda_init_bias: float = -6.0, theta_init: float = math.pi / 2, eps: float = 1e-6,
                 head_norm_mode: str = "full", rope_interleaved: bool = True):
        super().__init__()
        if embed_dim % num_heads != 0:
            raise ValueError("embed_dim must be divisible by num_heads.")
        if num_heads % num_kv_heads != 0:
            raise ValueError("num_heads must be divisible by num_kv_heads (GQA constraint).")
        self.embed_dim = embed_dim
        self.num_heads = num_heads
        self.num_kv_heads = num_kv_heads
        self.head_dim = embed_dim // num_heads
        if self.head_dim % 2 != 0:
            raise ValueError("head_dim must be even (required by RoPE + pairwise rotations).")
        self.q_proj = nn.Linear(embed_dim, num_heads * self.head_dim, bias=False)
        self.k_proj = nn.Linear(embed_dim, num_kv_heads * self.head_dim, bias=False)
        self.v_proj = nn.Linear(embed_dim, num_kv_heads * self.head_dim, bias=False)
        self.theta = nn.Parameter(torch.full((num_heads, self.head_dim // 2), theta_init))
        self.lambda_proj = nn.Linear(embed_dim, num_heads, bias=True)
        nn.init.constant_(self.lambda_proj.bias, lambda_init_bias)
        self.rope = RotaryEmbedding(self.head_dim, base=rope_base)
        self.head_norm_mode = head_norm_mode
        if head_norm_mode == "full":
            self.head_norm = HeadwiseRMSNorm(self.head_dim, eps=eps)
        elif head_norm_mode == "identity":
            self.head_norm = nn.Identity()
        else:
            raise ValueError(f"head_norm_mode must be 'full' or 'identity', got {head_norm_mode!r}")
        self.rope_interleaved = bool(rope_interleaved)
        self.o_proj = nn.Linear(num_heads * self.head_dim, embed_dim, bias=False)
        self._eps = float(eps)

    def attention_core(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, lam: torch.Tensor,
                       rope_cos: Optional[torch.Tensor], rope_sin: Optional[torch.Tensor], *, causal: int,
                       out: Optional[torch.Tensor] = None) -> torch.Tensor:
        """q (B,H,Lq,Dh) pre-RoPE (tables given) or post-RoPE; k, v
        (B,Hkv,Lk,Dh) post-RoPE; lam (B,H,Lq); causal 0 / 1 (lower-right) /
        2 (upper-left).  Returns head outputs (B, Lq, H, Dh)."""
        B, H, Lq, Dh = q.shape
        if out is None:
            out = torch.empty((B, Lq, H, Dh), dtype=q.dtype, device=q.device)
        ct = torch.cos(self.theta).to(dtype=q.dtype).contiguous()
        st = torch.sin(self.theta).to(dtype=q.dtype).contiguous()
        w = self.head_norm.weight.detach().to(q.dtype).contiguous() if self.head_norm_mode == "full" else None
        d = ops.bounded_attention(
            q=q, rope_cos=rope_cos, rope_sin=rope_sin, rope_interleaved=self.rope_interleaved, theta_cos=ct,
            theta_sin=st, k_prefix=None, v_prefix=None, allowed=None, k_block=k, v_block=v, lam=lam,
            rms_weight=w, eps=self._eps, out=out.permute(0, 2, 1, 3), causal=causal)
        return out

    def forward(self, x: torch.Tensor, *, is_causal: bool = True, attention_mask: Optional[torch.Tensor] = None,
                past_key_value: Optional[Tuple[torch.Tensor, torch.Tensor]] = None
                ) -> Tuple[torch.Tensor, Tuple[torch.Tensor, torch.Tensor]]:
        """x (B, L, D) -> (y, (k_total, v_total)) (baseline.py:95-147)."""
        if self.training:
            raise NotImplementedError("CoDAGQA on MI355X is inference-only (no backward kernels); call .eval()")
        if attention_mask is not None:
            raise NotImplementedError("explicit attention masks are not supported by the MI355X kernels")
        _hip.require_device(x)
        B, L, D = x.shape
        H, Hkv, Dh = self.num_heads, self.num_kv_heads, self.head_dim
        if past_key_value is not None:
            rows = self._decode_rows(x, past_key_value, is_causal)
            if rows is not None:
                return self._decode(x, rows, *past_key_value)
        q = self.q_proj(x).view(B, L, H, Dh).permute(0, 2, 1, 3)
        k = self.k_proj(x).view(B, L, Hkv, Dh).permute(0, 2, 1, 3)
        v = self.v_proj(x).view(B, L, Hkv, Dh).permute(0, 2, 1, 3)
        offset = past_key_value[0].size(2) if past_key_value is not None else 0
        cos, sin = self._rope_tables(offset, L, x.device, q.dtype)
        k = apply_rope(k, cos, sin, interleaved=self.rope_interleaved)
        if past_key_value is not None:
            k = torch.cat([past_key_value[0], k], dim=2)
            v = torch.cat([past_key_value[1], v], dim=2)
        else:
            v = v.contiguous()
        lam = torch.sigmoid(self.lambda_proj(x)).permute(0, 2, 1)
        # torch SDPA's is_causal aligns upper-left; with no past it is square
        heads = self.attention_core(q, k, v, lam, cos, sin, causal=2 if is_causal else 0)
        return self.o_proj(heads.view(B, L, D)), (k, v)

    def _decode_rows(self, x: torch.Tensor, past: Tuple[torch.Tensor, torch.Tensor], is_causal: bool):
        """The parameters' addresses (_front_rows) where _decode serves this
        call, else None: few new tokens on top of a past, no mask, bf16, at
        most 8 / G tokens a sequence, row-aligned K / V of the layer's shape
        whose planes stay within the kernel's 31-bit offsets."""
        B, L, _ = x.shape
        k, v = past
        if is_causal or L == 0 or x.dtype != torch.bfloat16 or k.dtype != x.dtype or v.dtype != x.dtype or \
                2 * L * (self.num_heads // self.num_kv_heads) > 16 or self.head_dim not in (32, 64, 128):
            return None
        shape = (B, self.num_kv_heads, k.shape[2] if k.dim() == 4 else 0, self.head_dim)
        st = k.stride()
        if not (tuple(k.shape) == shape and tuple(v.shape) == shape and shape[2] > 0 and v.stride() == st and
                st[3] == 1 and not (st[0] % 8 or st[1] % 8 or st[2] % 8) and
                0 <= st[2] and (shape[2] + L + 16) * max(st[2], self.head_dim) < 1 << 30 and
                not (k.data_ptr() % 16 or v.data_ptr() % 16) and k.device == v.device == x.device and
                not (torch.is_grad_enabled() and (k.requires_grad or v.requires_grad))):
            return None
        return self._front_rows(x)

    def _decode(self, x: torch.Tensor, rows: tuple, k_past: torch.Tensor, v_past: torch.Tensor):
        """forward() on top of a past for a few new tokens: one launch for the
        projections, the RoPE of k and the angle tables (coda_project_params),
        one for the attention and the concatenated K / V (coda_attn_append,
        which reads the past once for both), the merge of its splits, and
        o_proj; all on the parameters as they stand at the call."""
        B, L, D = x.shape
        H, Hkv, Dh = self.num_heads, self.num_kv_heads, self.head_dim
        past, M, e, half = k_past.shape[2], B * L, x.element_size(), Dh // 2
        lib, stream, dev = _hip.lib(), _hip.stream_of(x), x.device
        xs = _aligned(x)
        w = self.head_norm.weight.detach().to(x.dtype).contiguous() if self.head_norm_mode == "full" else None
        a = _hip.AttnDesc()
        a.dtype = _hip.dtype_code(x.dtype)
        a.B, a.H, a.Hkv, a.Lq, a.Dh = B, H, Hkv, L, Dh
        # q | k | v | lambda | gate of the new tokens, RoPE cos | sin, theta
        # cos | sin in one buffer
        sizes = [M * D * e, M * Hkv * Dh * e, M * Hkv * Dh * e, M * H * e, M * 4, L * half * e, L * half * e,
                 H * half * e, H * half * e]
        at = [0]
        for n in sizes:
            at.append(at[-1] + -(-n // 256) * 256)
        buf = torch.empty(at[-1], dtype=torch.uint8, device=dev)
        heads = torch.empty((B, L, D), dtype=x.dtype, device=dev)
        k, v = (torch.empty((B, Hkv, past + L, Dh), dtype=x.dtype, device=dev) for _ in range(2))
        q_p, k_p, v_p, l_p, g_p, rc_p, rs_p, tc_p, ts_p = (buf.data_ptr() + o for o in at[:-1])
        p = self._proj_params(rows)
        angles, th, keep = self._angles_rows(dev, past, L), self.theta, ()
        if angles is not None:
            p.inv_freq, p.inv_dtype = angles
            p.p0, p.rope_cos, p.rope_sin = past, rc_p, rs_p
        else:
            keep = self._rope_tables(past, L, dev, x.dtype)
            rc_p, rs_p = (t.data_ptr() for t in keep)
        if th.dtype in (torch.float32, torch.bfloat16) and th.device == dev and th.shape == (H, half) and \
                th.is_contiguous():
            p.theta, p.theta_dtype, p.theta_cos, p.theta_sin = th.data_ptr(), _hip.dtype_code(th.dtype), tc_p, ts_p
        else:
            tt = tuple(f(th).to(dtype=x.dtype).contiguous() for f in (torch.cos, torch.sin))
            tc_p, ts_p = (t.data_ptr() for t in tt)
            keep += tt
        d = self._proj_desc(x, M, L)
        d.rope_cos, d.rope_sin = rc_p, rs_p
        d.x, d.x_sm = xs.data_ptr(), D
        d.q, d.q_sm, d.k, d.k_sm, d.v, d.v_sm = q_p, D, k_p, Hkv * Dh, v_p, Hkv * Dh
        d.lam, d.lam_sm, d.g = l_p, H, g_p
        _hip.check(lib.coda_project_params(d, p, stream))
        a.q, a.q_sb, a.q_sh, a.q_sl = q_p, L * D, Dh, D
        a.theta_cos, a.theta_sin = tc_p, ts_p
        a.rope_cos, a.rope_sin, a.rope_interleaved = rc_p, rs_p, int(self.rope_interleaved)
        a.kp, a.vp, a.Lp = k_p, v_p, L
        a.p_sb, a.p_sh, a.p_sl = L * Hkv * Dh, Dh, Hkv * Dh
        a.kb, a.vb, a.Lb = k_past.data_ptr(), v_past.data_ptr(), past
        a.b_sb, a.b_sh, a.b_sl = k_past.stride()[:3]
        a.causal = 0
        a.lam, a.lam_sb, a.lam_sh, a.lam_sl = l_p, L * H, 1, H
        a.rms_w, a.eps, a.sm_scale = _hip.ptr(w), self._eps, 1.0 / math.sqrt(Dh)
        a.out, a.o_sb, a.o_sh, a.o_sl = heads.data_ptr(), L * D, Dh, D
        need = ctypes.c_size_t(0)
        _hip.check(lib.coda_attn_workspace_bytes(a, need))
        ws = torch.empty(need.value, dtype=torch.uint8, device=dev) if need.value else None
        a.workspace, a.workspace_bytes = _hip.ptr(ws), need.value
        _hip.check(lib.coda_attn_append(a, k.data_ptr(), v.data_ptr(), Hkv * (past + L) * Dh, (past + L) * Dh, Dh,
                                        stream))
        return self._out_rows(heads), (k, v)
