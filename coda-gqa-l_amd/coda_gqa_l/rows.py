"""Few-row projections shared by the bounded and unbounded layers: the packed
weights, RoPE rows and descriptors of coda_project_rows / coda_linear_rows
(csrc/proj.hip) for decode-shaped inputs."""

from __future__ import annotations

from typing import Optional, Tuple

import torch
import torch.nn as nn

from . import _hip
from .primitives import RotaryEmbedding


class _Made:
    """Where device tensors kept across calls were written: a use on another
    stream waits for them and keeps their memory from its allocator's reuse
    until that stream is past the use (under capture the caller's warm-up has
    ordered them, and neither is allowed)."""

    def __init__(self, *tensors: torch.Tensor):
        self.tensors = tensors
        self.stream, self.event = _hip.stream_of(tensors[0]), None
        if not torch.cuda.is_current_stream_capturing():
            self.event = torch.cuda.Event()
            self.event.record(torch.cuda.current_stream(tensors[0].device))

    def use(self) -> None:
        if self.event is None:
            return
        cur = torch.cuda.current_stream(self.tensors[0].device)
        if cur.cuda_stream != self.stream and not torch.cuda.is_current_stream_capturing():
            cur.wait_event(self.event)
            for t in self.tensors:
                t.record_stream(cur)


class RowsMixin:
    """Needs q_proj, k_proj, v_proj, lambda_proj, o_proj, rope, num_heads,
    num_kv_heads, head_dim, embed_dim and rope_interleaved; a write gate where
    _has_gate() says so."""

    def _has_gate(self) -> bool:
        return getattr(self, "write_policy", "none") != "none"

    def _derived(self, name: str, src: torch.Tensor, key, fn) -> torch.Tensor:
        """Tensor derived from a parameter, recomputed only when the parameter
        changes (in-place version counter or storage), so a decode step
        launches no conversion kernels."""
        cache = self.__dict__.setdefault("_derived_cache", {})
        tag = (src._version, src.data_ptr(), src.dtype, src.device)
        hit = cache.get((name, key))
        if hit is not None and hit[0] == tag:
            return hit[1]
        with torch.no_grad():
            val = fn()
        cache[(name, key)] = (tag, val)
        return val

    def _rope_rows(self, p0: int, L: int, device, dtype: torch.dtype) -> Tuple[torch.Tensor, torch.Tensor]:
        """RoPE tables (L, Dh/2) of positions p0 .. p0 + L - 1: rows of one
        cached table, grown by doubling; every element is the same fp32
        product and cos / sin as in a table made for these positions alone."""
        cache = self.__dict__.setdefault("_rope_cache", {})
        made = self.__dict__.setdefault("_rope_made", {})
        key = (torch.device(device), dtype)
        tab = cache.get(key)
        need = int(p0) + int(L)
        inv = self.rope.inv_freq
        hit = made.get(key)
        if tab is None or tab[0].shape[0] < need or hit is None or hit[0] is not inv or \
                hit[1] != (inv._version, inv.data_ptr()):
            n = 1 << max(12, (need - 1).bit_length())
            c, s_ = self.rope(seq_len=n, offset=0, device=device, dtype=dtype)
            tab = cache[key] = (c.contiguous(), s_.contiguous())
            made[key] = (inv, (inv._version, inv.data_ptr()), _Made(*tab) if tab[0].is_cuda else None)
        elif hit[2] is not None:
            hit[2].use()
        return tab[0][p0:need], tab[1][p0:need]

    def _rope_tables(self, p0: int, L: int, device, dtype: torch.dtype) -> Tuple[torch.Tensor, torch.Tensor]:
        """RoPE tables (L, Dh/2) of a prompt: rows of the cached table (made
        for the call alone they are seven small kernels, 20 us, and 45 us of
        host time), but for positions past 65536 (tables of at most 32 MiB
        are kept), under capture (a graph must not hold rows of a table that
        a later call replaces) and where self.rope is not the plain module."""
        r = self.rope
        if p0 + L > 65536 or type(r) is not RotaryEmbedding or r._forward_hooks or r._forward_pre_hooks or \
                nn.modules.module._has_any_global_hook() or torch.cuda.is_current_stream_capturing():
            c, s_ = r(seq_len=L, offset=p0, device=device, dtype=dtype)
            return c.contiguous(), s_.contiguous()
        return self._rope_rows(p0, L, device, dtype)

    def _proj_pack(self, dtype: torch.dtype):
        """Packed [q | k | v | lambda | write] weights (n_feat, D) in `dtype`,
        float32 biases (zero for a linear without one) and the weights'
        layout code for coda_project, per parameter version; with half-split
        RoPE each k head's rows are reordered to the pairs (i, i + Dh/2) on
        adjacent rows.  On a HIP device the weights are kept in the row
        kernel's fragment tiles (coda_rows_pack, layout 1)."""
        gate = self._has_gate()
        lins = (self.q_proj, self.k_proj, self.v_proj, self.lambda_proj) + ((self.write_proj,) if gate else ())
        ps = [t for lin in lins for t in (lin.weight, lin.bias) if t is not None]
        tag = tuple((t._version, t.data_ptr(), t.dtype, t.device) for t in ps) + (self.rope_interleaved,)
        cache = self.__dict__.setdefault("_derived_cache", {})
        hit = cache.get(("proj", dtype))
        if hit is not None and hit[0] == tag:
            made = self.__dict__.get("_proj_made", {}).get(dtype)
            if made is not None:
                made.use()
            return hit[1]
        H, Hkv, Dh = self.num_heads, self.num_kv_heads, self.head_dim
        with torch.no_grad():
            dev = self.q_proj.weight.device
            wk, bk = self.k_proj.weight, self.k_proj.bias
            if not self.rope_interleaved:
                half = Dh // 2
                pair = torch.stack([torch.arange(half), torch.arange(half) + half], 1).reshape(-1)
                perm = (torch.arange(Hkv)[:, None] * Dh + pair[None]).reshape(-1).to(dev)
                wk = wk[perm]
                bk = bk[perm] if bk is not None else None
            ws = [self.q_proj.weight, wk, self.v_proj.weight, self.lambda_proj.weight]
            bt = [self.q_proj.bias, bk, self.v_proj.bias, self.lambda_proj.bias]
            if gate:
                ws.append(self.write_proj.weight)
                bt.append(self.write_proj.bias)
            b = torch.cat([t.detach().float() if t is not None else torch.zeros(wt.shape[0], device=dev)
                           for t, wt in zip(bt, ws)])
            b = torch.cat([b, torch.zeros((-b.numel()) % 4, device=dev)])
            ws = [t.detach().to(dtype) for t in ws]
            if ws[0].is_cuda:
                w, layout = self._rows_tiles(*ws), 1
            else:
                w, layout = torch.cat(ws).contiguous(), 0
        val = (w, b.contiguous(), layout)
        cache[("proj", dtype)] = (tag, val)
        if w.is_cuda:
            self.__dict__.setdefault("_proj_made", {})[dtype] = _Made(*val[:2])
        return val

    @staticmethod
    def _rows_tiles(*parts: torch.Tensor) -> torch.Tensor:
        """(n, D) weights, the parts one after the other, in the row kernel's
        fragment tiles (coda_rows_pack), n rounded up to a multiple of 64.  A
        part that starts on a row block of 16 is packed from where it is (a
        layer's first token paid a concatenation of all its weights
        otherwise: 340 MB of traffic and a second buffer at 10305 x 8192);
        rows that the loads of the kernel can't take are copied first."""
        groups, n = [], 0
        for t in parts:
            if n % 16:
                groups[-1].append(t)
            else:
                groups.append([t])
            n += t.shape[0]
        D, rows = parts[0].shape[1], -(-n // 64) * 64
        # (each launch pads its rows to 64 and the next one writes over the
        # padding; the last one's may end past `rows`)
        wt = torch.empty((rows + 64, D), dtype=parts[0].dtype, device=parts[0].device)
        wt[n // 64 * 64:].zero_()
        at, fn, dt, stream = 0, _hip.lib().coda_rows_pack, _hip.dtype_code(wt.dtype), _hip.stream_of(wt)
        for g in groups:
            w = g[0].contiguous() if len(g) == 1 else torch.cat(g)
            if w.data_ptr() % 16:
                w = w.clone()
            _hip.check(fn(dt, w.data_ptr(), w.shape[0], D, D, wt[at:].data_ptr(), stream))
            at += w.shape[0]
        return wt[:rows]

    @staticmethod
    def _plain_call(x: torch.Tensor, *lins: nn.Module) -> bool:
        """Whether calling these modules on x is no more than their matrix
        product: nn.Linear in x's dtype, no hooks, no autocast, no gradient."""
        if torch.is_autocast_enabled(x.device.type) or nn.modules.module._has_any_global_hook():
            return False
        grad = torch.is_grad_enabled()
        if grad and x.requires_grad:
            return False
        for m in lins:
            if type(m) is not nn.Linear or m.weight.dtype != x.dtype or m._forward_hooks or m._forward_pre_hooks or \
                    grad and m.weight.requires_grad:
                return False
        return True

    def _out_rows(self, heads: torch.Tensor) -> torch.Tensor:
        """o_proj of decode-shaped heads (B, L, H*Dh): at most 32 token rows
        through the row kernel (bf16 4096 x 4096: 8.1 us at 1 row and 11.1 at
        32 against 12.0 and 12.4 for the library's GEMM, which is ahead at 64
        with 12.8 against 14.5).  Smaller bf16 layers take it up to 64 rows
        (2048 x 2048) and 128 (1024 x 1024): the step waits for the host there
        and this way is the shorter one (a token of 40 rows, 1024 x 1024: 32.6
        us against 44.4 through the library)."""
        B, L, K = heads.shape
        o = self.o_proj
        most = 32
        if heads.dtype == torch.bfloat16 and type(o) is nn.Linear and o.weight.numel() <= 1 << 22:
            most = 128 if o.weight.numel() <= 1 << 20 else 64
        if B * L > most or K % 64 or heads.dtype not in (torch.bfloat16, torch.float32) or \
                not self._plain_call(heads, o) or not heads.is_contiguous():
            return o(heads)
        w, bias = o.weight, o.bias
        tag = (w._version, w.data_ptr(), w.dtype, w.device) + (() if bias is None else (bias._version, bias.data_ptr()))
        hit = self.__dict__.get("_o_rows")
        if hit is None or hit[0] != tag:
            with torch.no_grad():
                tiles = self._rows_tiles(w.detach())
                b = None if bias is None else bias.detach().float().contiguous()
            hit = self.__dict__["_o_rows"] = (tag, tiles, b, _Made(*(t for t in (tiles, b) if t is not None)))
        hit[3].use()
        y = torch.empty((B, L, o.out_features), dtype=heads.dtype, device=heads.device)
        _hip.check(_hip.lib().coda_linear_rows(
            _hip.dtype_code(heads.dtype), heads.data_ptr(), K, B * L, hit[1].data_ptr(), o.out_features, K, _hip.ptr(hit[2]),
            y.data_ptr(), o.out_features, _hip.stream_of(heads)))
        return y

    def _proj_desc(self, x: torch.Tensor, M: int, L: int, cos: torch.Tensor, sin: torch.Tensor):
        d = _hip.ProjDesc()
        d.dtype, d.M, d.D, d.L = _hip.dtype_code(x.dtype), M, self.embed_dim, L
        d.H, d.Hkv, d.Dh = self.num_heads, self.num_kv_heads, self.head_dim
        d.rope_interleaved, d.gate = int(self.rope_interleaved), int(self._has_gate())
        d.rope_cos, d.rope_sin = cos.data_ptr(), sin.data_ptr()
        return d

    def _fused_front_ok(self, x: torch.Tensor) -> bool:
        """Whether coda_project_rows serves x: D a multiple of 64, head_dim a
        multiple of 4, and few token rows.  bf16: at most 64, or 128 (5 library
        GEMMs with their sigmoids and RoPE take 103 us at 10305 x 8192 and 128
        rows, the one launch 53); fp32: at most 32 (at 64 the library's GEMMs
        are ahead)."""
        B, L, D = x.shape
        if D % 64 or self.head_dim % 4:
            return False
        if x.dtype == torch.bfloat16 and B * L <= 64:
            return True
        most = 128 if x.dtype == torch.bfloat16 else 32 if x.dtype == torch.float32 else 0
        gate = (self.write_proj,) if self._has_gate() else ()
        return B * L <= most and self._plain_call(x, self.q_proj, self.k_proj, self.v_proj, self.lambda_proj, *gate)
