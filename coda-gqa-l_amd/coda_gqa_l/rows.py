"""Few-row projections shared by the bounded and unbounded layers: parameters
(as they lie, or packed), RoPE tables and descriptors of the row kernels
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
        if not _capturing():
            self.event = torch.cuda.Event()
            self.event.record(torch.cuda.current_stream(tensors[0].device))

    def use(self) -> None:
        if self.event is None:
            return
        cur = torch.cuda.current_stream(self.tensors[0].device)
        if cur.cuda_stream != self.stream and not _capturing():
            cur.wait_event(self.event)
            for t in self.tensors:
                t.record_stream(cur)


def _capturing() -> bool:
    return torch.cuda.is_initialized() and torch.cuda.is_current_stream_capturing()


def _version(t: torch.Tensor) -> Optional[int]:
    """t's in-place version; None for an inference tensor, which counts none."""
    try:
        return t._version
    except RuntimeError:
        return None


def _aligned(x: torch.Tensor) -> torch.Tensor:
    """x, or a copy of it where the row kernels can't read it in place
    (contiguous() returns a contiguous x off a 16-byte address as it is)."""
    return x if x.is_contiguous() and x.data_ptr() % 16 == 0 else x.clone(memory_format=torch.contiguous_format)


# What a layer keeps between calls: copies derived from parameters; and
# workspaces, plans and buffers
_PARAM_COPIES = ("_derived_cache", "_rope_cache", "_rope_made", "_proj_made", "_fast", "_dplan")
_KEPT = _PARAM_COPIES + ("_graph_held", "_step_ws_bytes", "_route_ws", "_route_tag", "_ws_cache", "_block_ws",
                         "_block_checked", "_status_pending", "_snap_cache", "_last_chunk_group")


class RowsMixin:
    """Needs q_proj, k_proj, v_proj, lambda_proj, o_proj, rope, num_heads,
    num_kv_heads, head_dim, embed_dim and rope_interleaved; a write gate where
    _has_gate() says so."""

    def __getstate__(self) -> dict:
        """For copies and saves of the layer: without what it keeps between
        calls (events and descriptors that can't travel, addresses that would
        name the original's memory)."""
        return {k: v for k, v in self.__dict__.items() if k not in _KEPT}

    def drop_parameter_copies(self) -> None:
        """Forget everything derived from parameters: for after a change of
        one that torch does not count (through .data, or from outside torch).
        Counted changes need no such call.  Prompts, unbounded layers, o_proj,
        fp32 steps and steps of more than 64 rows read the projections' own
        values in any case; kept are the packed q / k / v / lambda / gate
        weights and RoPE rows of bf16 steps of up to 64 rows, and a bounded
        layer's noise angles, head norm weight and summary rates."""
        for k in _PARAM_COPIES:
            self.__dict__.pop(k, None)

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
            return self._handed(hit[1])
        with torch.no_grad():
            val = fn()
        if not _capturing():
            cache[(name, key)] = (tag, val)
        return val

    def _handed(self, val):
        """val, a tensor or several kept across calls, on its way to a caller:
        under capture it stays alive with the layer (a graph goes on reading
        it when the layer has replaced it).  What is made under capture is not
        kept at all: nothing has run yet."""
        if _capturing():
            held = self.__dict__.setdefault("_graph_held", {})
            held[id(val)] = val
        return val

    def _rope_rows(self, p0: int, L: int, device, dtype: torch.dtype) -> Tuple[torch.Tensor, torch.Tensor]:
        """RoPE tables (L, Dh/2) of positions p0 .. p0 + L - 1: rows of one
        cached table, grown by doubling; every element is the same fp32
        product and cos / sin as in a table made for these positions alone.
        (Not under capture: a larger table replaces and frees it.)"""
        cache = self.__dict__.setdefault("_rope_cache", {})
        made = self.__dict__.setdefault("_rope_made", {})
        key = (torch.device(device), dtype)
        tab = cache.get(key)
        need = int(p0) + int(L)
        inv = getattr(self.rope, "inv_freq", None)  # (a module of the user's own may have none)
        tag, hit = None if inv is None else (_version(inv), inv.data_ptr()), made.get(key)
        if tab is None or tab[0].shape[0] < need or hit is None or hit[0] is not self.rope or hit[1] is not inv or \
                hit[2] != tag:
            n = 1 << max(12, (need - 1).bit_length())
            c, s_ = self.rope(seq_len=n, offset=0, device=device, dtype=dtype)
            tab = cache[key] = (c.contiguous(), s_.contiguous())
            made[key] = (self.rope, inv, tag, _Made(*tab) if tab[0].is_cuda else None)
        elif hit[3] is not None:
            hit[3].use()
        return tab[0][p0:need], tab[1][p0:need]

    def _rope_tables(self, p0: int, L: int, device, dtype: torch.dtype) -> Tuple[torch.Tensor, torch.Tensor]:
        """RoPE tables (L, Dh/2): made for the call, by one launch in place of
        the module's seven where the module is the plain one (nothing is kept,
        so nothing can go stale, be freed under a captured graph or be read
        before it is written)."""
        a = None
        if dtype in (torch.float32, torch.bfloat16) and not nn.modules.module._has_any_global_hook():
            a = self._angles_rows(device, p0, L)
        if a is None:
            c, s_ = self.rope(seq_len=L, offset=p0, device=device, dtype=dtype)
            return c.contiguous(), s_.contiguous()
        half = self.head_dim // 2
        c, s_ = torch.empty((L, half), dtype=dtype, device=device), torch.empty((L, half), dtype=dtype, device=device)
        _hip.check(_hip.lib().coda_rope_tables(_hip.dtype_code(dtype), a[0], a[1], p0, L, half, c.data_ptr(),
                                               s_.data_ptr(), _hip.stream_of(c)))
        return c, s_

    def _proj_pack(self, dtype: torch.dtype):
        """Packed [q | k | v | lambda | write] weights (n_feat, D) in `dtype`,
        float32 biases (zero for a linear without one) and the weights'
        layout code for coda_project, per parameter version; with half-split
        RoPE each k head's rows are reordered to the pairs (i, i + Dh/2) on
        adjacent rows.  On a HIP device the weights are kept in the row
        kernel's fragment tiles (layout 1), made in one launch where they have
        that dtype already."""
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
            return self._handed(hit[1])
        H, Hkv, Dh, D = self.num_heads, self.num_kv_heads, self.head_dim, self.embed_dim
        sizes = (H * Dh, Hkv * Dh, Hkv * Dh, H, 1)
        for lin, n in zip(lins, sizes):
            if tuple(lin.weight.shape) != (n, D) or lin.bias is not None and tuple(lin.bias.shape) != (n,):
                raise RuntimeError(f"projection weight {tuple(lin.weight.shape)} is not ({n}, {D})")
        n_feat = sum(sizes[:len(lins)])
        dev, layout = self.q_proj.weight.device, 0
        if all(t.is_cuda and t.device == dev and t.dtype == dtype and t.stride(-1) == 1 for t in ps):
            w, layout = torch.empty((-(-n_feat // 64) * 64, D), dtype=dtype, device=dev), 1
            b = torch.empty(-(-n_feat // 4) * 4, dtype=torch.float32, device=dev)
            d, rows = self._proj_desc(w, 0, 1), []
            for lin in lins:
                rows += (lin.weight.data_ptr(), lin.weight.stride(0), _hip.ptr(lin.bias))
            _hip.check(_hip.lib().coda_project_pack_params(d, self._proj_params(rows), w.data_ptr(), b.data_ptr(),
                                                           _hip.stream_of(w)))
        else:
            with torch.no_grad():
                ws, bs = [lin.weight.detach() for lin in lins], []
                for lin in lins:
                    bs.append(lin.bias.detach().float() if lin.bias is not None
                              else torch.zeros(lin.out_features, device=dev))
                if not self.rope_interleaved:
                    pair = torch.stack([torch.arange(Dh // 2), torch.arange(Dh // 2) + Dh // 2], 1).reshape(-1)
                    perm = (torch.arange(Hkv)[:, None] * Dh + pair[None]).reshape(-1).to(dev)
                    ws[1], bs[1] = ws[1][perm], bs[1][perm]
                w = torch.cat(ws).to(dtype).contiguous()
                b = torch.cat(bs + [torch.zeros((-n_feat) % 4, device=dev)])
                if w.is_cuda:
                    tiles, layout = torch.empty((-(-n_feat // 64) * 64, D), dtype=dtype, device=dev), 1
                    _hip.check(_hip.lib().coda_rows_pack(_hip.dtype_code(dtype), w.data_ptr(), n_feat, D, D,
                                                         tiles.data_ptr(), _hip.stream_of(w)))
                    w = tiles
        val = (w, b, layout)
        if w.is_cuda and _capturing():
            return val
        cache[("proj", dtype)] = (tag, val)
        if w.is_cuda:
            self.__dict__.setdefault("_proj_made", {})[dtype] = _Made(*val[:2])
        return val

    def _packed_weights(self, x: torch.Tensor):
        """_proj_pack for x's projections: the kernel reads x's device alone."""
        val = self._proj_pack(x.dtype)
        if val[0].device != x.device:
            raise RuntimeError(f"projection weights on {val[0].device}, input on {x.device}")
        return val

    def _plain_rows(self, x: torch.Tensor, *names: str) -> Optional[tuple]:
        """(address, row stride, bias address) of each of these linears' own
        parameters, one after the other, where calling the module on x is no
        more than its matrix product and the row kernels can take that: an
        nn.Linear in x's dtype on x's device, no hooks, no forward of the
        instance's own or put in the class's place, no autocast, no gradient,
        no tensor subclass.  Else None.  Asked at every call: nothing about a
        parameter is remembered."""
        if torch.is_autocast_enabled(x.device.type) or nn.modules.module._has_any_global_hook() or \
                type(x) not in (torch.Tensor, nn.Parameter) or nn.Linear.forward.__module__ != "torch.nn.modules.linear":
            return None
        grad = torch.is_grad_enabled()
        if grad and x.requires_grad:
            return None
        dt, dev, K, mods, out = x.dtype, x.device, x.shape[-1], self._modules, []
        for name in names:
            m = mods[name]
            d = m.__dict__
            if type(m) is not nn.Linear or m._forward_hooks or m._forward_pre_hooks or "forward" in d:
                return None
            ps = d["_parameters"]
            w, b = ps.get("weight"), ps.get("bias")
            if type(w) is not nn.Parameter or w.dtype is not dt or w.device != dev or w.dim() != 2:
                return None
            n, k = w.shape
            if k != K or n != m.out_features or w.stride(1) != 1 or w.stride(0) < K or grad and w.requires_grad:
                return None
            pb = None
            if b is not None:
                if type(b) is not nn.Parameter or b.dtype is not dt or b.device != dev or b.shape != (n,) or \
                        b.stride(0) != 1 or grad and b.requires_grad:
                    return None
                pb = b.data_ptr()
            out += (w.data_ptr(), w.stride(0), pb)
        return tuple(out)

    def _out_rows(self, heads: torch.Tensor, kept: bool = False) -> torch.Tensor:
        """o_proj of decode-shaped heads (B, L, H*Dh): few token rows of not too
        large a layer through the row kernel, on the parameter itself.  kept:
        the caller writes over heads later, so a module that may hold on to
        its input (hooks, autograd) gets a copy.

        The kernel against the library's GEMM, us, bf16: 4096 x 4096 8.7 and
        14.9 at 1 row, 12.9 and 12.7 at 32, 16.2 and 14.4 at 64; 2048 x 2048
        4.2 and 5.2, 6.3 and 7.3 at 64; 1024 x 1024 3.1 and 4.2, 6.6 and 6.5
        at 64, 10.3 and 5.2 at 128, where the step still waits for the host
        and this way is the shorter one (a token of 128 rows 39.9 us among
        others and 71.5 alone against 54.1 and 71.8 through the module); 8192
        x 8192 29.4 and 28.9 at 1 row, 31.5 and 28.8 at 16: the library's.
        fp32: 1024 x 1024 4.5 and 5.5 at 1 row, 5.8 and 6.8 at 32; a token of
        32 rows, 2048 x 2048, 53.5 us against 61.1; 4096 x 4096 15.8 and 15.4
        at 1 row, 22.8 and 18.5 at 32: the library's."""
        B, L, K = heads.shape
        o = self.o_proj
        rows, most = B * L, 0
        if type(o) is nn.Linear:
            n = o.out_features * K
            if heads.dtype == torch.bfloat16:
                most = 128 if n <= 1 << 20 else 64 if n <= 1 << 22 else 32 if n <= 1 << 24 else 0
            elif heads.dtype == torch.float32:
                most = 32 if n <= 1 << 22 else 0
        fits = 0 < rows <= most and K % 64 == 0 and heads.is_contiguous()
        p = self._plain_rows(heads, "o_proj") if fits or kept else None
        if p is None or not fits:
            return o(heads.clone() if kept and p is None else heads)
        y = torch.empty((B, L, o.out_features), dtype=heads.dtype, device=heads.device)
        _hip.check(_hip.lib().coda_linear_params(
            _hip.dtype_code(heads.dtype), heads.data_ptr(), K, rows, p[0], p[1], o.out_features, K, p[2], y.data_ptr(),
            o.out_features, _hip.stream_of(heads)))
        return y

    def _proj_desc(self, x: torch.Tensor, M: int, L: int, cos: Optional[torch.Tensor] = None,
                   sin: Optional[torch.Tensor] = None):
        d = _hip.ProjDesc()
        d.dtype, d.M, d.D, d.L = _hip.dtype_code(x.dtype), M, self.embed_dim, L
        d.H, d.Hkv, d.Dh = self.num_heads, self.num_kv_heads, self.head_dim
        d.rope_interleaved, d.gate = int(self.rope_interleaved), int(self._has_gate())
        d.rope_cos, d.rope_sin = _hip.ptr(cos), _hip.ptr(sin)
        return d

    def _packed_front_ok(self, x: torch.Tensor) -> bool:
        """Whether the front end on packed weights serves x: bf16, at most 64
        token rows, D a multiple of 64, head_dim a multiple of 4.  (6177 x
        4096, weights not in cache: 12.2 us at 1 row and 18.2 at 64, on the
        parameters 13.3 and 22.3; 10305 x 8192 31.3 against 36.1.)"""
        B, L, D = x.shape
        return x.dtype == torch.bfloat16 and B * L <= 64 and D % 64 == 0 and self.head_dim % 4 == 0 and \
            D == self.embed_dim

    def _front_rows(self, x: torch.Tensor) -> Optional[tuple]:
        """The parameters' addresses (_plain_rows) where coda_project_params
        serves x: D a multiple of 64, head_dim a multiple of 4, and few token
        rows.  bf16: at most 128 (5 library GEMMs with their sigmoids and
        RoPE take 103 us at 10305 x 8192 and 128 rows, this launch 64); fp32: at most 32 (at
        64 the library's GEMMs are ahead)."""
        B, L, D = x.shape
        most = 128 if x.dtype == torch.bfloat16 else 32 if x.dtype == torch.float32 else 0
        if not 0 < B * L <= most or D % 64 or D != self.embed_dim or self.head_dim % 4:
            return None
        names = ("q_proj", "k_proj", "v_proj", "lambda_proj")
        p = self._plain_rows(x, *names, *(("write_proj",) if self._has_gate() else ()))
        if p is None:
            return None
        H, F, mods = self.num_heads, self.num_heads * self.head_dim, self._modules
        Fk = self.num_kv_heads * self.head_dim
        if tuple(mods[n].out_features for n in names) != (F, Fk, Fk, H) or \
                self._has_gate() and mods["write_proj"].out_features != 1:
            return None
        return p

    def _fused_front_ok(self, x: torch.Tensor) -> bool:
        """Whether one launch of the row kernel serves x's projections."""
        return self._packed_front_ok(x) or self._front_rows(x) is not None

    def _angles_rows(self, device, p0: int, L: int) -> Optional[tuple]:
        """(address, type code) of the RoPE frequencies where the kernels can
        make the tables of positions p0 .. p0 + L - 1 as self.rope would."""
        r = self._modules["rope"]
        if type(r) is not RotaryEmbedding or r._forward_hooks or r._forward_pre_hooks or "forward" in r.__dict__ or \
                not 0 <= p0 <= (1 << 24) - L:
            return None
        inv = r._buffers.get("inv_freq")
        if inv is None or inv.dtype not in (torch.float32, torch.bfloat16) or inv.device != device or \
                inv.shape != (self.head_dim // 2,) or inv.stride(0) != 1:
            return None
        return inv.data_ptr(), _hip.dtype_code(inv.dtype)

    @staticmethod
    def _proj_params(rows: tuple) -> "_hip.ProjParams":
        p = _hip.ProjParams()
        for i in range(len(rows) // 3):
            p.w[i], p.w_sm[i], p.b[i] = rows[3 * i:3 * i + 3]
        return p
