"""UV-50M forward for inference on the HIP kernels: int8 KV state, one decode step for a ragged batch, packed prefill.

Mirrors ultraviolet/kernels/fast_decode.py of the reference (KernelDecodeState :21-57, decode_step_fast :272-334,
_prefill_packed / prefill_packed_host :117-269) and the layer math of ultraviolet/model.py (Attention.qkv / post
:302-335, Block.finish :567-571, MathLM.logits :824-827).  The projections of a 16-bit engine run on this
library's GEMMs with the norms, residual updates and the SwiGLU in them (_pass_kind), an fp32 engine's on the vendor library's; what lies
between them is one fused HIP kernel per stage, and K/V go straight into the cache.
One decode step is a fixed launch sequence with no host synchronisation: it reads per-row positions on the device, so
a single captured graph serves every context length (the reference needs one graph per 1024-token bucket,
model.py:1099-1100)."""
from __future__ import annotations

import ctypes as C
import weakref

import numpy as np
import torch
from torch import Tensor

from .. import _lib as L
from ..kernels.decode_attn import build_attn_args, build_fused_args, decode_attention, rope_table
from ..kernels.gemm import RESID, SOFTCAP, STORE, SWIGLU, gemm_args, gemm_supported, gemm_tn
from ..kernels.kv_quant import kv_write
from ..kernels.varlen_attn import packed_attention, packed_attention_args
from ..kernels.fused_sample import fused_sample_seeded, greedy_sample
from .config import UVConfig
from .plan import Guard, PassPlan, launch
from .weights import UVWeights


class KVState:
    """Slot-indexed KV cache (reference: KernelDecodeState, fast_decode.py:21-57): per layer k, v (B, K, S, hd) int8
    and k_scale, v_scale (B, K, S) fp16 with S = max_len, rounded up to a multiple of 32, on global layers and min(window, max_len)
    on local (ring) layers; pos / starts (B,) int64 on the device.  pos is the next position to write.  kv_dtype "fp16" (the
    reference's name for "unquantized") keeps k, v in `dtype`, the activation type, with no scales.  These tensors are all there
    is: a ring holds the last S positions, also where the global caches have room for a few more."""

    def __init__(self, cfg: UVConfig, B: int, max_len: int, device="cuda", kv_dtype: str = "int8", dtype=torch.bfloat16):
        # Global caches have S rounded up to 32 slots: the MFMA attention kernel streams 32-key tiles and needs S % 4 == 0 for its
        # 8-byte scale loads (other S fall back to the generic kernel).  Rings keep their length: a window, or what a short max_len
        # cuts it to (short_ring).
        self.local_len = min(cfg.window, max_len)
        max_len = (max_len + 31) // 32 * 32
        self.cfg, self.B, self.max_len = cfg, B, max_len
        assert kv_dtype in ("int8", "fp16") and (kv_dtype == "int8" or dtype in (torch.float16, torch.bfloat16))
        self.kv_dtype, self.quantized = kv_dtype, kv_dtype == "int8"
        cdt = torch.int8 if self.quantized else dtype
        dev = torch.device(device)
        self.k, self.v, self.k_scale, self.v_scale = [], [], [], []
        for l in range(cfg.n_layers):
            S = max_len if cfg.is_global(l) else self.local_len
            shp = (B, cfg.n_kv_heads, S, cfg.head_dim)
            self.k.append(torch.zeros(shp, dtype=cdt, device=dev))
            self.v.append(torch.zeros(shp, dtype=cdt, device=dev))
            self.k_scale.append(torch.zeros(shp[:3], dtype=torch.float16, device=dev) if self.quantized else None)
            self.v_scale.append(torch.zeros(shp[:3], dtype=torch.float16, device=dev) if self.quantized else None)
        self.pos = torch.zeros(B, dtype=torch.long, device=dev)
        self.starts = torch.zeros(B, dtype=torch.long, device=dev)

    def cache(self, l: int) -> tuple:
        """k, v, k_scale, v_scale of layer l."""
        return self.k[l], self.v[l], self.k_scale[l], self.v_scale[l]

    def slots(self, l: int) -> int:
        """Slots of layer l's rows (of its k; the launch checks the rest)."""
        return self.k[l].size(2)

    def short_ring(self, l: int) -> bool:
        """Whether layer l's cache is a ring that max_len cut below the window to a length of no whole tiles.  The engine runs those
        as any_ring launches: the generic kernel, which takes such lengths too, needs 133 us where they need 5.2 on 16 rows of
        up to 128 keys, and they keep its precision.  (Windows of such a length stay on the generic kernel.)"""
        S = self.slots(l)
        return not self.cfg.is_global(l) and 32 <= S < self.cfg.window and S % 32 != 0

    def window(self, l: int) -> int:
        """Keys that layer l attends (0: all): no more than its ring holds."""
        return 0 if self.cfg.is_global(l) else min(self.cfg.window, self.slots(l)) if self.short_ring(l) else self.cfg.window

    def nbytes(self) -> int:
        return sum(t.numel() * t.element_size() for t in self.k + self.v + self.k_scale + self.v_scale if t is not None)

    @torch.no_grad()
    def copy_rows(self, src: Tensor, dst: Tensor, upto: int):
        """Cache rows dst <- cache rows src for the first `upto` slots of every layer, with pos and starts (src, dst: (n,)
        int64 on the device).  A sequence's cache depends only on its own tokens and quantisation is per row, so a prompt
        shared by several sequences is prefilled once and copied: the copies hold the bytes their own prefill would write."""
        for l in range(self.cfg.n_layers):
            for t in self.cache(l):
                if t is not None:
                    n = min(upto, t.size(2))
                    t[dst, :, :n] = t[src, :, :n]
        self.pos[dst] = self.pos[src]
        self.starts[dst] = self.starts[src]


def kv_bytes_per_seq(cfg: UVConfig, ctx: int) -> int:
    """int8 cache bytes of one sequence at context ctx (reference: fast_decode.py:64-67)."""
    per_pos = 2 * cfg.n_kv_heads * (cfg.head_dim + 2)
    return sum(per_pos * (ctx if cfg.is_global(l) else min(ctx, cfg.window)) for l in range(cfg.n_layers))


def rms_norm_eps(dtype: torch.dtype) -> float:
    """eps that torch.nn.functional.rms_norm(x, eps=None) uses for this dtype in the installed torch (the reference relies
    on that default, model.py:190-191): machine epsilon of the dtype in some releases, of fp32 in others.  Probed once on
    the CPU with a vector small enough that the two candidates give clearly different results."""
    x = torch.full((8,), 2.0 ** -6, dtype=dtype)
    y = float(torch.nn.functional.rms_norm(x, (8,)).float()[0])
    cands = [float(torch.finfo(dtype).eps), float(torch.finfo(torch.float32).eps)]
    refs = [2.0 ** -6 / (2.0 ** -12 + e) ** 0.5 for e in cands]
    return cands[int(np.argmin([abs(y - r) for r in refs]))]


class _Stage:
    """A pinned host buffer that launches read in place, and the event behind the last of them.  The allocator does not know
    of such readers, so the buffer waits for them before it goes."""

    buf = event = None

    def wait(self):
        if self.event is not None:
            self.event.synchronize()

    def __del__(self):
        try:
            self.wait()
        except Exception:   # the runtime is already gone (interpreter exit)
            pass


def _swiglu_norm(b: dict, h: Tensor, n: int, dt_code: int, cfg: UVConfig, eps: float):
    """UVEngine._swiglu_norm on the engine's buffers b."""
    rc = L.lib().uvmi_swiglu_norm(b["gu"].data_ptr(), h.data_ptr(), dt_code, n, cfg.d_ff, cfg.d_model, eps, b["act"].data_ptr(), L.stream_ptr(h))
    L.check(rc, "uvmi_swiglu_norm")


class UVEngine:
    def __init__(self, weights: UVWeights, max_tokens: int, skinny_rows: int = 192, fold_qkv_rows: int = 1 << 30, fold_o_rows: int = 1 << 30,
                 fold_gu_rows: int = 1 << 30, lean: bool = True, fold: bool = True, gemm_config: int = 0,
                 tiled_prefill: bool = True, big_rows: int = 12288, fold_down_rows: tuple = (0, 5120), general_skinny_rows: int = 384, oproj_rows: int | None = None):
        """max_tokens: largest number of token rows one forward call processes (decode rows + packed prefill tokens).
        skinny_rows: decode passes of at most this many rows run every projection on this library's GEMM, the residual updates out of
        place (general_skinny_rows: the same for passes of the plain path); fold_qkv_rows, fold_o_rows,
        fold_gu_rows: above skinny_rows, row counts up to which the QKV projection (with the pre-norm), the output
        projection (with the residual update) and the gate-up projection (with the pre-norm and the SwiGLU) run on this
        library's GEMM kernels instead of the vendor library's (see _trunk_folded); lean / fold: the launch plans that drop
        the residual-add and norm launches (off: the general path); gemm_config: form of the hand-written GEMM (0: its own
        choice by size; tests force the tiled forms at a few rows); big_rows: passes of the general path with at least this
        many rows (a packed prefill, a mixed pass) run the down projection too on this library's GEMM, whose 256 x 256 tile
        form is as fast as the vendor library there; fold_down_rows: (first, last) row count of passes whose down projection runs
        on this library's GEMM; oproj_rows: decode passes of at most this many rows leave the output projection and its residual
        update to the attention launch (None: as many as it takes, 0: none).  The defaults are measured on
        UV-50M (between fold_down_rows and big_rows the vendor library's down projection is up to 14 % the faster below ~7000 rows and within
        6 % of this library's, either way, from there on)."""
        self.w, self.cfg = weights, weights.cfg
        cfg, dt, dev = self.cfg, weights.dtype, weights.device
        assert cfg.head_dim == 64, "the fused kernels are written for head_dim 64"
        self.dtype, self.device, self.max_tokens = dt, dev, max_tokens
        self.dt_code = L.dtype_code(dt)
        self.eps = rms_norm_eps(dt)
        # the attention kernels' query operand: the activation type; an fp32 engine keeps fp32 queries, which run on the plain
        # fp32 attention kernel (no 16-bit rounding of q or of the probabilities anywhere on its path)
        self.q_dtype = dt
        n, d, H, K, hd, f = max_tokens, cfg.d_model, cfg.n_heads, cfg.n_kv_heads, cfg.head_dim, cfg.d_ff
        e = lambda *s, dtype=dt: torch.empty(*s, dtype=dtype, device=dev)
        self.buf = dict(x=e(n, d), xn=e(n, d), h=e(n, d), qkv=e(n, (H + 2 * K) * hd), q=e(n, H, hd, dtype=self.q_dtype),
                        k=e(n, K, hd), v=e(n, K, hd), zg=e(n, H * hd), a=e(n, d), gu=e(n, 2 * f), act=e(n, f), m=e(n, d),
                        vhat=e(n, K, hd, dtype=torch.float32), gate=e(n, H, dtype=torch.float32))
        # decode steps of a 16-bit engine take q, k, v and the gate logits from one extended projection and leave the
        # post-processing to the attention kernel (one launch less per layer)
        self.fuse_qkv = dt in (torch.bfloat16, torch.float16) and cfg.n_heads // cfg.n_kv_heads <= 8 and cfg.n_pairs in (0, 16)
        self.qkvx_keep = None
        # Decode passes of at most this many rows keep the block's two hiddens apart (h and x); above it the folded plan updates
        # one in place.
        self.skinny_rows = int(skinny_rows) if dt in (torch.bfloat16, torch.float16) else 0
        # Of those, passes of at most this many rows have the output projection in the attention launch (one launch of five less a layer:
        # a step of 1 row 191 -> 173 us, of 8 204 -> 186, of 16 203 -> 188, of 32 214 -> 201, to the same bits).
        one_kv = cfg.n_heads == 8 and cfg.n_kv_heads == 1 and self.skinny_rows > 0
        most = L.lib().uvmi_attn_oproj_rows(cfg.d_model) if one_kv else 0
        self.oproj_rows = most if oproj_rows is None else min(int(oproj_rows), most)
        # passes of the plain path run on this library's GEMM up to this many rows: their alternative is the vendor library with
        # separate SwiGLU and norm launches
        self.general_skinny_rows = int(general_skinny_rows) if dt in (torch.bfloat16, torch.float16) else 0
        # above skinny_rows: row counts up to which the QKV, output and gate-up projections run on this library's GEMM
        self.fold_qkv_rows = int(fold_qkv_rows)
        self.fold_o_rows, self.fold_gu_rows = int(fold_o_rows), int(fold_gu_rows)
        self.lean, self.fold, self.gemm_config = bool(lean), bool(fold), int(gemm_config)
        self.tiled_prefill = bool(tiled_prefill)
        self.big_rows = int(big_rows)
        # the down projection runs on this library's GEMM between these row counts (per launch 5.9 against the vendor library's
        # 8.5 us at 512 rows, 13.5 against 14.2 at 3072, 19.3 against 19.9 at 4608, 21.6 against 19.3 at 6144)
        self.fold_down_rows = (int(fold_down_rows[0]), int(fold_down_rows[1]))
        self.head_own_rows = 288       # decode steps of at most this many rows run the head GEMM on this library's kernel (own_head_ok)
        self.hidden_is_raw = False
        self._new_scratch()
        self._rope_tabs: dict[int, Tensor] = {}  # rotation tables by position count, kept for the engine's life (graphs hold them)
        if self.fuse_qkv:
            self.buf["qkvx"] = e(n, UVWeights.qkv_ext_rows(cfg))
        self.pf_ws = torch.empty(L.lib().uvmi_prefill_attn_workspace_bytes(n), dtype=torch.uint8, device=dev)  # fails now if the library is missing

    def _new_scratch(self):
        """What belongs to this object and this process, and no copy takes along: staging memory and recorded passes."""
        self._stage, self._stage_at = [_Stage() for _ in range(2)], 0   # (_staging)
        self._plans = weakref.WeakKeyDictionary()   # per state its recorded passes (_planned), for as long as it lives
        self._rec = None               # the PassPlan being recorded (None: operations are launched as they come)

    def __getstate__(self):
        return {k: v for k, v in self.__dict__.items() if k not in ("_stage", "_stage_at", "_plans", "_rec")}

    def __setstate__(self, d):
        self.__dict__.update({"oproj_rows": 0, **d})   # (an engine saved before it had them: five launches a layer, as it ran then)
        self._new_scratch()

    # ------------------------------------------------------------------------------------------------ kernels
    # An operation is launched at once and, while a plan is being recorded (_planned), appended to it, where the names given for its
    # fields say which per-call values they hold: n the token rows of the pass, tok / pos / rows / last / starts / cu the
    # addresses of its arrays, Np / nd the prompt tokens and decode rows of a mixed pass, *_d addresses of its decode part.
    def _op(self, kind: int, args, keep=(), **per_call):
        launch(kind, args, L.stream_ptr(self.buf["x"]))
        if self._rec is not None:
            self._rec.op(kind, args, keep, **per_call)

    def _lib_gemm(self, n: int, fn):
        """A GEMM of the vendor library on the first n rows of the engine's buffers: fn(n), which does not hold the engine (a
        recorded list keeps it, and the engine keeps the lists)."""
        fn(n)
        if self._rec is not None:
            self._rec.call(lambda values: fn(values["n"]))

    def _gemm(self, a: Tensor, w: Tensor, out: Tensor, epilogue: int = STORE, **kw):
        g = gemm_args(a, w, out, epilogue, **kw)
        self._op(L.OP_GEMM_RESID if epilogue == RESID else L.OP_GEMM, g, (a, w, out), M="n")

    def _gemm_sums(self, a: Tensor, w: Tensor, out: Tensor, epilogue: int = STORE, **kw):
        """_gemm of a pass that keeps its hidden's sums of squares (_sums_ok), in what buf h is for other plans."""
        g = gemm_args(a, w, out, epilogue, **kw)
        self._op(L.OP_GEMM_SUMS, L.GemmSumsArgs(C.addressof(g), *self._sums()), (g, a, w, out, self.buf["h"]))
        if self._rec is not None:
            self._rec.field(g, "M", "n")

    def _sums(self) -> tuple[int, int]:
        return self.buf["h"].data_ptr(), (self.max_tokens + 3) // 4 * 4

    def _sums_ok(self, n: int) -> bool:
        """Whether the residual updates of a packed pass sum the squares of the hidden they write for the projections that take its norm.
        Formed again in every tile that reads it, it is a sixteenth of their matrix instructions: gate-up at 18 432 rows 86 us against 79 so, extended
        projection 22.7 / 21.4; at 33 216 rows 144 / 133, 37.7 / 35.9; the updates pay 0.4 - 1 us each (a pass of 64 prompts 2252 -> 2200 us, a
        mixed one 3901 -> 3824).  All four have to run on the kernels of many rows (uvmi_gemm_sums' rule: the updates' two contractions are over the
        heads' columns and over d_ff)."""
        cfg = self.cfg
        return (n >= max(self.big_rows, 12288) and n <= min(self.fold_qkv_rows, 1 << 16) and self.gemm_config == 0 and 256 <= cfg.d_model <= 1024
                and cfg.n_heads * cfg.head_dim >= 128 and cfg.d_ff >= 128)

    def _embed_norm(self, tok: Tensor, n: int):
        b = self.buf
        self._op(L.OP_NORM, L.NormArgs(x=self.w.embed.data_ptr(), tok=tok.data_ptr(), vocab=self.cfg.vocab_size, dtype=self.dt_code, rows=n,
                                       d=self.cfg.d_model, eps=self.eps, h_out=b["x"].data_ptr(), n_out=b["xn"].data_ptr()),
                 (self.w.embed, tok), rows="n", tok="tok")

    def _add_norm(self, x: Tensor, y: Tensor, a: float, bb: float, n: int, h_out: Tensor | None, n_out: Tensor, advance: Tensor | None = None):
        """h_out = a x + bb y, n_out = its norm; advance: positions of the rows to count up in the same launch."""
        args = L.NormArgs(x=x.data_ptr(), y=y.data_ptr(), dtype=self.dt_code, a=a, b=bb, rows=n, d=self.cfg.d_model, eps=self.eps,
                          h_out=None if h_out is None else h_out.data_ptr(), n_out=n_out.data_ptr(),
                          advance=None if advance is None else advance.data_ptr())
        self._op(L.OP_NORM, args, (), rows="n", **({} if advance is None else {"advance": "pos"}))

    def _qkv_post(self, l: int, tok: Tensor, pos: Tensor, rows: Tensor | None, last_pos: Tensor | None, st: KVState | None,
                  n: int, write_cache: bool = True, ext: bool = False, gemm=None, sums: bool = False):
        """ext: the rows come from the extended projection (buf qkvx), whose last columns are the gates' logits: the
        normalised block input is then not read.  gemm: the argument block of that projection, which has yet to be made: the two
        are one operation; sums: with the rows' norm from the sums that the residual update before it left (_gemm_sums)."""
        cfg, b, W = self.cfg, self.buf, self.w.layers[l]
        glob = cfg.is_global(l)
        a = L.QkvPostArgs()
        a.qkv, a.dtype, a.xn = b["qkvx" if ext else "qkv"].data_ptr(), self.dt_code, b["xn"].data_ptr()
        if ext:
            a.qkv_ld, a.ext_logits = b["qkvx"].stride(0), 1
        has_ve = cfg.has_ve(l)
        per_call = dict(n="n", pos="pos")
        if has_ve:
            a.ve_table, a.ve_gate, a.tok = self.w.value_embed.data_ptr(), W["ve_gate"].data_ptr(), tok.data_ptr()
            per_call["tok"] = "tok"
        a.pos = pos.data_ptr()
        if rows is not None:
            a.rows = rows.data_ptr()
            per_call["rows"] = "rows"
        if last_pos is not None:
            a.last_pos = last_pos.data_ptr()
            per_call["last_pos"] = "last"
        a.inv_freq = self.w.inv_freq.data_ptr()
        a.q_out, a.q_dtype = b["q"].data_ptr(), L.dtype_code(self.q_dtype)
        a.k_out, a.v_out = b["k"].data_ptr(), b["v"].data_ptr()
        write_cache = st is not None and write_cache
        fused_write = write_cache and self._append_fused(st)
        if fused_write:   # int8 codes and scales, or (a cache of the activation type) the values as they are
            kc, vc, ks, vs = st.cache(l)
            a.k_cache, a.v_cache, a.S = kc.data_ptr(), vc.data_ptr(), kc.size(2)
            a.scb, a.sch, a.scs = kc.stride(0), kc.stride(1), kc.stride(2)
            if st.quantized:
                a.k_scale, a.v_scale, a.ssb, a.ssh = ks.data_ptr(), vs.data_ptr(), ks.stride(0), ks.stride(1)
        a.n, a.vocab = n, cfg.vocab_size
        a.H, a.KH, a.hd, a.d, a.ve_ch, a.n_pairs = cfg.n_heads, cfg.n_kv_heads, cfg.head_dim, cfg.d_model, cfg.ve_gate_channels, cfg.n_pairs
        a.ring, a.has_ve = int(not glob), int(has_ve)
        a.rope = int(((not glob) or cfg.global_rope) and cfg.n_pairs > 0)
        if a.rope and st is not None:   # cos / sin from the table of the state's positions instead of per-token cosf / sinf
            tab = self.rope_table(st.max_len)
            a.rope_table, a.rope_positions = tab.data_ptr(), tab.size(0)
        a.eps = self.eps
        if cfg.xsa:
            a.vhat_out, a.xsa_eps = b["vhat"].data_ptr(), float(cfg.xsa_eps)
        if W["attn_gate"] is not None:
            a.gate_w, a.gate_ch, a.gate_out = W["attn_gate"].data_ptr(), cfg.gate_ch, b["gate"].data_ptr()
        keep = (tok, pos, rows, last_pos)
        if gemm is None:
            self._op(L.OP_QKV_POST, a, keep, **per_call)
        else:
            self._op(L.OP_QKV_PROJ, L.QkvProjArgs(C.addressof(gemm), C.addressof(a), *(self._sums() if sums else (None, 0))), (gemm, a, keep, b["h"]))
            if self._rec is not None:
                self._rec.field(gemm, "M", "n")
                for field, name in per_call.items():
                    self._rec.field(a, field, name)
        if write_cache and not fused_write:
            self._write_kv_cast(l, pos, rows, last_pos, st, n)

    def _append_fused(self, st: KVState) -> bool:
        """Whether the post-processing kernel appends to this state's caches (int8, or unquantized in the activation type)."""
        return st.quantized or st.k[0].dtype == self.dtype

    def _write_kv_cast(self, l: int, pos: Tensor, rows: Tensor | None, last_pos: Tensor | None, st: KVState, n: int):
        """Unquantized caches of another type than the activations: buf k / v of the n rows go, cast, to slot pos (pos % S on a
        ring) of their cache rows - the two kv_write calls of the reference's step (fast_decode.py:291-294, 315-317).
        Dropped, as the fused append drops them: padding rows, positions past a linear cache, and prompt positions a ring
        will not keep (older than last_pos - S)."""
        cfg, b = self.cfg, self.buf
        K = cfg.n_kv_heads
        kc, vc = st.cache(l)[:2]
        S = kc.size(2)
        ring = not cfg.is_global(l)
        row = torch.arange(n, device=pos.device) if rows is None else rows[:n]
        p = pos[:n]
        slot = torch.remainder(p, S) if ring else p
        ok = (row >= 0) & (p >= 0) & (slot < S)
        if ring and last_pos is not None:
            ok &= p > last_pos[:n] - S
        flat = (row[:, None] * K + torch.arange(K, device=pos.device)[None, :]) * S + slot[:, None]
        flat = torch.where(ok[:, None], flat, torch.full_like(flat, -1)).reshape(-1).contiguous()
        kv_write(kc, None, flat, b["k"][:n])
        kv_write(vc, None, flat, b["v"][:n])

    def _attn_post(self, l: int, z: Tensor, n: int, off: int = 0):
        """XSA + gate of rows off..off+n of the call (z holds just those rows); writes buf zg[off:off+n]."""
        cfg, b, W = self.cfg, self.buf, self.w.layers[l]
        rc = L.lib().uvmi_attn_post(z.data_ptr(), L.dtype_code(z.dtype), b["v"][off:].data_ptr(), b["xn"][off:].data_ptr(), self.dt_code,
                                    None if W["attn_gate"] is None else W["attn_gate"].data_ptr(),
                                    None if W["xsa"] is None else W["xsa"].data_ptr(), float(cfg.xsa_eps), n, cfg.n_heads,
                                    cfg.n_kv_heads, cfg.head_dim, cfg.d_model, cfg.gate_ch, b["zg"][off:].data_ptr(), L.stream_ptr(z))
        L.check(rc, "uvmi_attn_post")

    def _finish_attn(self, l: int, z, h: Tensor | None = None):
        """What an attention (the attn of _trunk) left undone: XSA + gate of the rows it returned.  The gate is a product of the
        block's normalised input, buf xn; h: the block's input, where a plan has not written its norm there."""
        parts = [(off, z) for off, z in (z if isinstance(z, list) else [(0, z)]) if z is not None and z.size(0)]
        if parts and h is not None and self.w.layers[l]["attn_gate"] is not None:
            self._add_norm(h, h, 1.0, 0.0, h.size(0), None, self.buf["xn"])
        for off, z in parts:
            self._attn_post(l, z, z.size(0), off)

    def _swiglu(self, n: int):
        b = self.buf
        rc = L.lib().uvmi_swiglu(b["gu"].data_ptr(), self.dt_code, n, self.cfg.d_ff, b["act"].data_ptr(), L.stream_ptr(b["gu"]))
        L.check(rc, "uvmi_swiglu")

    def _swiglu_norm(self, h: Tensor, n: int):
        """buf act = SwiGLU of rmsnorm(h) @ gu.T, from buf gu = h @ gu.T (the norm as a row scale of the product)."""
        _swiglu_norm(self.buf, h, n, self.dt_code, self.cfg, self.eps)

    # ------------------------------------------------------------------------------------------------ trunk
    def cache_attention_plannable(self, l: int, st: KVState) -> bool:
        """Whether layer l's attention over the cache is one launch with the fused XSA + gate epilogue: the MFMA kernel streams
        32-key tiles (rings need S % 32 == 0 or to be short ones, linear int8 caches S % 4 == 0) and serves
        int8 caches and caches in the q dtype."""
        cfg, S = self.cfg, st.slots(l)
        mfma_cache = self.q_dtype != torch.float32 and (st.quantized or st.k[l].dtype == self.q_dtype)
        return (mfma_cache and cfg.xsa and cfg.n_heads // cfg.n_kv_heads <= 8 and S >= 32
                and (S % (4 if cfg.is_global(l) else 32) == 0 or st.short_ring(l)))

    def cache_attention(self, l: int, q: Tensor, st: KVState, pos: Tensor, starts: Tensor, n: int, rows: Tensor | None = None,
                        off: int = 0):
        """Decode attention of layer l over the cache (int8, or unquantized) with the fused XSA + gate epilogue for the n rows that sit at
        off..off+n of the call's buffers (q is already that slice); writes buf zg[off:off+n] and returns None, or, where
        the fused epilogue does not apply, returns the plain attention output for _attn_post."""
        cfg, b, W = self.cfg, self.buf, self.w.layers[l]
        glob, window = cfg.is_global(l), st.window(l)
        if self.cache_attention_plannable(l, st) and q.dtype == self.q_dtype:
            if rows is not None:
                rows = rows.to(pos.dtype).contiguous()
            out = b["zg"][off:off + n].view(n, cfg.n_heads, cfg.head_dim)
            gate = None if W["attn_gate"] is None else b["gate"][off:off + n]
            k, v, ks, vs = st.cache(l)
            a, keep = build_attn_args(q, k, v, pos.contiguous(), starts.contiguous(), cfg.attn_scale, window, not glob, ks, vs, 1, out, 0, rows,
                                      (b["vhat"][off:off + n], gate, W["xsa"], out.dtype), any_ring=st.short_ring(l))
            self._op(L.OP_DECODE_ATTN, a, (keep, q, pos, starts), B="nd", q="q_d", post_vhat="vhat_d", out="zg_d", pos="pos_d", starts="starts_d",
                     **({} if gate is None else {"post_gate": "gate_d"}), **({} if rows is None else {"rows": "rows_d"}))
            return None
        k, v, ks, vs = st.cache(l)
        return decode_attention(q, k, v, pos, starts, cfg.attn_scale, num_splits=1, window=window, ring=not glob, k_scale=ks, v_scale=vs, rows=rows)

    def prompt_attention_plannable(self) -> bool:
        """Whether the packed prompts' attention is one launch with the fused XSA + gate epilogue (16-bit engine)."""
        cfg = self.cfg
        return (cfg.xsa and self.dtype in (torch.bfloat16, torch.float16) and self.q_dtype == self.dtype and cfg.head_dim == 64
                and cfg.n_heads // cfg.n_kv_heads <= 8)

    def prompt_attention(self, l: int, q: Tensor, N: int, cu: Tensor, gemm=None):
        """Causal (windowed on local layers) attention of the N packed prompt tokens at the head of the call's buffers over
        their own unquantized K / V (buf k, v).  Where the MFMA kernel runs (16-bit engine) XSA and the gate ride in its
        epilogue - it writes buf zg[:N] and None is returned; otherwise the plain attention output is returned for
        _attn_post.  The segment table of cu is built by layer 0's call and reused by the other layers of the pass.  gemm: the argument
        block of the output projection of buf zg (prompt_attention_plannable passes without decode rows): the two are one operation."""
        cfg, b, W = self.cfg, self.buf, self.w.layers[l]
        w = 0 if cfg.is_global(l) else cfg.window
        if self.prompt_attention_plannable():
            if N == 0:
                return None
            out = b["zg"][:N].view(N, cfg.n_heads, cfg.head_dim)
            a = packed_attention_args(q, b["k"][:N], b["v"][:N], cu, cfg.attn_scale, w, out, self.pf_ws, segments_ready=l > 0,
                                      post=(b["vhat"][:N], None if W["attn_gate"] is None else b["gate"][:N], W["xsa"]))
            per_call = dict(N="Np", cu_seqlens="cu", n_seg="n_seg")
            if gemm is None:
                self._op(L.OP_PREFILL_ATTN, a, (q, out, cu), **per_call)
            else:
                self._op(L.OP_PREFILL_ATTN_O, L.PrefillAttnOArgs(C.addressof(a), C.addressof(gemm)), (gemm, a, q, out, cu))
                if self._rec is not None:
                    self._rec.field(gemm, "M", "n")
                    for field, name in per_call.items():
                        self._rec.field(a, field, name)
            return None
        return packed_attention(q, b["k"][:N], b["v"][:N], cu, cfg.attn_scale, w, workspace=self.pf_ws, segments_ready=l > 0)

    def fused_layer_ok(self, l: int, st: KVState) -> bool:
        """Whether layer l's decode attention can take the fused path: the MFMA kernel streams 32-key tiles."""
        S = st.slots(l)
        return self.fuse_qkv and (st.quantized or st.k[l].dtype == self.dtype) and S >= 32 and (S % 32 == 0 or st.short_ring(l))

    def _fused_layers_ok(self, st: KVState) -> bool:
        """fused_layer_ok of every layer.  (Asked on every step, so the common answer takes one short walk: 3 us less.)"""
        if self.fuse_qkv and st.quantized and not any(S % 32 or S < 32 for S in {k.size(2) for k in st.k}):
            return True
        return all(self.fused_layer_ok(l, st) for l in range(self.cfg.n_layers))

    def rope_table(self, n_positions: int) -> Tensor:
        """cos / sin of every position below n_positions in the activation type's rounding, built once per size."""
        t = self._rope_tabs.get(n_positions)
        if t is None:
            if torch.cuda.is_current_stream_capturing():
                raise RuntimeError("the rotation table must exist before a graph is captured: call rope_table(state.max_len) first")
            t = self._rope_tabs[n_positions] = rope_table(self.w.inv_freq, n_positions, self.dtype)
        return t

    def _fuse_dict(self, l: int, tok: Tensor, st: KVState) -> dict:
        cfg = self.cfg
        glob = cfg.is_global(l)
        has_ve = cfg.has_ve(l)
        rope = ((not glob) or cfg.global_rope) and cfg.n_pairs > 0
        return dict(ext_col=(cfg.n_heads + 2 * cfg.n_kv_heads) * cfg.head_dim, has_gate=cfg.gate_ch > 0, tok=tok if has_ve else None,
                    ve_table=self.w.value_embed if has_ve else None, vocab=cfg.vocab_size, rope_table=self.rope_table(st.max_len) if rope else None,
                    n_pairs=cfg.n_pairs, rope=rope, eps=self.eps, xsa_eps=cfg.xsa_eps)

    def fused_cache_attention(self, l: int, tok: Tensor, st: KVState, pos: Tensor, starts: Tensor, n: int, rows: Tensor | None = None,
                              oproj: bool = False):
        """Decode attention of layer l straight from buf qkvx (the extended projection of the n rows): QK-norm, rotation,
        value embedding, int8 append, attention over lo..pos, XSA and gate in one launch; writes buf zg.  oproj: also the output
        projection and the block's first residual update; writes buf h instead."""
        a, keep = self.fused_attention_args(l, self.buf["qkvx"], tok, st, pos, starts, n, rows, oproj)
        if self._rec is not None and self.cfg.has_ve(l):
            self._rec.field(keep[0][2], "tok", "tok")
        self._op(L.OP_DECODE_ATTN, a, (keep, pos, starts), B="n", pos="pos", starts="starts", **({} if rows is None else {"rows": "rows"}))

    def fused_attention_args(self, l: int, qkvx: Tensor, tok: Tensor, st: KVState, pos: Tensor, starts: Tensor, n: int,
                             rows: Tensor | None = None, oproj: bool = False):
        """The uvmi_attn_args struct fused_cache_attention launches for layer l, on a given copy of that layer's extended
        projection (qkvx_keep): lets a benchmark re-issue exactly the step's launches through the C ABI.  Re-issuing it
        on the step's own positions rewrites the same K/V bytes."""
        cfg, b, W = self.cfg, self.buf, self.w.layers[l]
        glob = cfg.is_global(l)
        out = b["zg"][:n].view(n, cfg.n_heads, cfg.head_dim)
        k, v, ks, vs = st.cache(l)
        fuse = self._fuse_dict(l, tok, st)
        if oproj:
            fuse["oproj"] = dict(w=W["wo"], resid=b["x"][:n], out=b["h"][:n], ca=W["resid_attn"], cb=W["post_attn"])
        return build_fused_args(qkvx[:n], cfg.n_heads, k, v, pos, starts, cfg.attn_scale, st.window(l), not glob, ks, vs, W["xsa"], out,
                                fuse, rows, any_ring=st.short_ring(l))

    def cache_attention_args(self, l: int, st: KVState, pos: Tensor, starts: Tensor, n: int, rows: Tensor | None = None):
        """The uvmi_attn_args struct cache_attention would launch for layer l on the engine's buffers (fused path only):
        lets a benchmark re-issue exactly the step's attention launches through the C ABI without the Python wrapper."""
        cfg, b, W = self.cfg, self.buf, self.w.layers[l]
        glob = cfg.is_global(l)
        out = b["zg"][:n].view(n, cfg.n_heads, cfg.head_dim)
        k, v, ks, vs = st.cache(l)
        return build_attn_args(b["q"][:n], k, v, pos, starts, cfg.attn_scale, st.window(l), not glob, ks, vs, 1, out, 0, rows,
                               (b["vhat"][:n], None if W["attn_gate"] is None else b["gate"][:n], W["xsa"], out.dtype), any_ring=st.short_ring(l))

    def _trunk(self, tok: Tensor, pos: Tensor, n: int, attn, rows=None, last_pos=None, st: KVState | None = None,
               fused_attn=None, defer_final_norm: bool = False, advance: bool = False, final_norm: bool = True, oproj: bool = False) -> Tensor:
        """n token rows through all layers; attn(l, q (n, H, hd)) -> z (n, H, hd), or None when it wrote the post-processed
        result to buf zg itself, or a list of (first row, z) of the parts that it left to _attn_post; it runs after K/V of the
        layer have been appended to the cache and written unquantized to buf k / v.  Returns the final normed hidden (n, d) (a
        buffer).  defer_final_norm: a plan whose last block leaves the hidden un-normalised returns it as it is and sets self.hidden_is_raw - the caller's head GEMM then carries the final
        norm as the row scale of its product (head_of), and the norm launch goes away; final_norm False: likewise at any row
        count, for a caller that norms the few rows it needs itself (_normed).  advance: the final norm's launch counts pos up
        by one.  oproj: attn(l, q, gemm) makes the output projection of the rows too (_layers_packed)."""
        cfg, b = self.cfg, self.buf
        assert n <= self.max_tokens
        self._embed_norm(tok, n)
        x, xn = b["x"][:n], b["xn"][:n]
        adv = pos if advance else None
        self.hidden_is_raw = False
        raw = True          # the last block leaves buf x un-normalised
        kind = self._pass_kind(n, fused_attn is not None, st)
        if kind in ("lean", "lean-o"):
            self._layers_lean(n, fused_attn, kind == "lean-o")
        elif kind == "folded":
            self._layers_folded(n, fused_attn)
        elif kind == "packed":
            self._layers_packed(n, tok, pos, rows, last_pos, st, attn, oproj)
        else:
            raw = self._layers_plain(n, tok, pos, rows, last_pos, st, attn, fused_attn)
        if raw:
            if not final_norm or (defer_final_norm and self.own_head_ok(n)):
                self.hidden_is_raw = True
                return x
            self._add_norm(x, x, 1.0, 0.0, n, None, b["xn"], adv)   # the final norm
        elif advance:
            pos.add_(1)
        return xn

    def _pass_kind(self, n: int, fused: bool, st: KVState | None) -> str:
        """The launch plan of a pass of n rows: "lean" ("lean-o": with the output projection in the attention launch) and "folded" for decode rows whose every layer takes the fused
        attention, "packed" for prompts, mixed passes and the unfused attention of a 16-bit engine, "plain" for the rest
        (fp32, widths the GEMMs do not take, plans switched off)."""
        cfg = self.cfg
        ok16 = self.dtype != torch.float32
        il = all("gu_il" in W for W in self.w.layers)
        div = cfg.d_model % 64 == 0 and (cfg.n_heads * cfg.head_dim) % 64 == 0
        if fused and ok16 and self._fused_layers_ok(st):
            skinny = n <= self.skinny_rows and div
            if skinny and self.lean and il and cfg.d_ff % 64 == 0:
                return "lean-o" if n <= self.oproj_rows else "lean"
            if self.fold and not skinny and cfg.d_ff % 8 == 0:
                return "folded"
        if not fused and ok16 and self.fold and self.tiled_prefill and self.fuse_qkv and il and div and cfg.d_ff % 64 == 0:
            return "packed"
        return "plain"

    def _keep_projection(self, l: int, n: int):
        if self.qkvx_keep is not None:   # a benchmark re-issues this layer's launch later on the same projection
            self.qkvx_keep[l][:n].copy_(self.buf["qkvx"][:n])

    def _project_qkv(self, l: int, n: int, own: bool = True, **kw):
        """buf qkvx = the extended projection (q, k, v and the gates' logits) of the n rows, with the block's pre-norm as the
        row scale of the product (layer 0: the embedding's norm exists already); own: on this library's GEMM."""
        b, W = self.buf, self.w.layers[l]
        if not own:
            if l > 0:
                self._add_norm(b["x"], b["x"], 1.0, 0.0, n, None, b["xn"])
            self._lib_gemm(n, lambda n: torch.mm(b["xn"][:n], W["wqkv_ext"].t(), out=b["qkvx"][:n]))
        elif l == 0:
            self._gemm(b["xn"][:n], W["wqkv_ext"], b["qkvx"][:n], **kw)
        else:
            self._gemm(b["x"][:n], W["wqkv_ext"], b["qkvx"][:n], norm_eps=self.eps, **kw)

    def _layers_lean(self, n: int, fused_attn, oproj: bool):
        """Decode passes of few rows: every projection on this library's GEMM, the residual updates in the epilogues of the output
        and down projections, both pre-norms as row scales of the products that read them.  Five launches per layer; four where
        the attention launch does the output projection and its residual update (oproj)."""
        b = self.buf
        x, h, zg, act = b["x"][:n], b["h"][:n], b["zg"][:n], b["act"][:n]
        for l, W in enumerate(self.w.layers):
            self._project_qkv(l, n)
            self._keep_projection(l, n)
            if oproj:
                fused_attn(l, oproj=True)
            else:
                fused_attn(l)
                self._gemm(zg, W["wo"], h, RESID, resid=x, ca=W["resid_attn"], cb=W["post_attn"])
            self._gemm(h, W["gu_il"], act, SWIGLU, norm_eps=self.eps)
            self._gemm(act, W["down"], x, RESID, resid=h, ca=W["resid_mlp"], cb=W["post_mlp"])

    def _layers_folded(self, n: int, fused_attn):
        """Decode passes of many rows, five launches per layer: QKV projection with the block's pre-norm as a row scale, fused
        attention, output projection with the residual update in place, gate-up projection with the MLP's pre-norm and the
        SwiGLU in its epilogue (the (n, 2 f) intermediate and the normalised hidden are never written), down projection with the
        residual update (the vendor library's C = alpha A B + beta C outside fold_down_rows)."""
        cfg, b = self.cfg, self.buf
        x, zg, act = b["x"][:n], b["zg"][:n], b["act"][:n]
        gc, dt_code, eps = self.gemm_config, self.dt_code, self.eps
        sk_ok = cfg.d_model % 64 == 0 and (cfg.n_heads * cfg.head_dim) % 64 == 0
        sk_qkv, sk_o = sk_ok and n <= self.fold_qkv_rows, sk_ok and n <= self.fold_o_rows
        for l, W in enumerate(self.w.layers):
            self._project_qkv(l, n, sk_qkv, config=gc)
            self._keep_projection(l, n)
            fused_attn(l)
            # x <- resid_attn * x + post_attn * (zg @ wo.T), in place (every element is read and written by the same lane)
            if sk_o:
                self._gemm(zg, W["wo"], x, RESID, resid=x, ca=W["resid_attn"], cb=W["post_attn"], config=gc)
            else:
                self._lib_gemm(n, lambda n, W=W: torch.addmm(b["x"][:n], b["zg"][:n], W["wo"].t(), beta=W["resid_attn"], alpha=W["post_attn"], out=b["x"][:n]))
            if sk_ok and "gu_il" in W and n <= self.fold_gu_rows:
                self._gemm(x, W["gu_il"], act, SWIGLU, norm_eps=self.eps, config=gc)
            else:
                def gate_up(n, W=W):
                    torch.mm(b["x"][:n], W["gu"].t(), out=b["gu"][:n])
                    _swiglu_norm(b, b["x"][:n], n, dt_code, cfg, eps)
                self._lib_gemm(n, gate_up)
            # x <- resid_mlp * x + post_mlp * (act @ down.T)
            self._down(l, n, sk_ok and self.fold_down_rows[0] <= n <= self.fold_down_rows[1] and cfg.d_ff % 64 == 0)

    def _down(self, l: int, n: int, own: bool):
        """x <- resid_mlp * x + post_mlp * (act @ down.T), in place."""
        b, W = self.buf, self.w.layers[l]
        if own:
            self._gemm(b["act"][:n], W["down"], b["x"][:n], RESID, resid=b["x"][:n], ca=W["resid_mlp"], cb=W["post_mlp"], config=self.gemm_config)
        else:
            self._lib_gemm(n, lambda n: torch.addmm(b["x"][:n], b["act"][:n], W["down"].t(), beta=W["resid_mlp"], alpha=W["post_mlp"], out=b["x"][:n]))

    def _layers_packed(self, n: int, tok, pos, rows, last_pos, st, attn, oproj: bool = False):
        """Prompts, mixed passes and the unfused attention of a 16-bit engine: the extended projection with the pre-norm in it,
        the post-processing kernel (which takes the gates' logits from the projection and appends to the cache), the
        attention launches, output and down projections with the residual update in place, gate-up with the pre-norm and
        the SwiGLU.  The normalised hidden is not written between blocks (_finish_attn forms it for a layer whose attention
        leaves its epilogue to _attn_post; layer 0 has the embedding's).  oproj: attn also takes the output projection (prompt_attention's gemm)."""
        cfg, b = self.cfg, self.buf
        x, zg, act = b["x"][:n], b["zg"][:n], b["act"][:n]
        gc = self.gemm_config
        own_down = n <= self.skinny_rows or n >= self.big_rows or self.fold_down_rows[0] <= n <= self.fold_down_rows[1]
        sums = last_pos is not None and self._sums_ok(n)
        project = self._gemm_sums if sums else self._gemm
        for l, W in enumerate(self.w.layers):
            gemm = None
            if n <= self.fold_qkv_rows and last_pos is not None:   # (decode rows alone: the projection of the fused attention's plans, to the same bits)
                gemm = gemm_args(b["xn" if l == 0 else "x"][:n], W["wqkv_ext"], b["qkvx"][:n], norm_eps=None if l == 0 else self.eps, config=gc)
            else:
                self._project_qkv(l, n, n <= self.fold_qkv_rows, config=gc)
            self._qkv_post(l, tok, pos, rows, last_pos, st, n, ext=True, gemm=gemm, sums=sums and l > 0)
            if oproj and not sums:   # (the attention's launch, or one behind it)
                attn(l, b["q"][:n], gemm_args(zg, W["wo"], x, RESID, resid=x, ca=W["resid_attn"], cb=W["post_attn"], config=gc))
            else:
                self._finish_attn(l, attn(l, b["q"][:n]), x if l > 0 else None)
                project(zg, W["wo"], x, RESID, resid=x, ca=W["resid_attn"], cb=W["post_attn"], config=gc)
            project(x, W["gu_il"], act, SWIGLU, norm_eps=self.eps, config=gc)
            if sums:
                self._gemm_sums(act, W["down"], x, RESID, resid=x, ca=W["resid_mlp"], cb=W["post_mlp"])
            else:
                self._down(l, n, own_down)

    def _layers_plain(self, n: int, tok, pos, rows, last_pos, st, attn, fused_attn) -> bool:
        """The reference's order of operations on the vendor library's GEMMs (16-bit passes of few rows: on this one's),
        one launch per step between them: fp32 engines, widths the other plans do not take.  Returns whether buf x was
        left un-normalised (else buf xn holds the final norm)."""
        cfg, b = self.cfg, self.buf
        x, xn = b["x"][:n], b["xn"][:n]
        skinny_rows = self.skinny_rows if fused_attn is not None else max(self.skinny_rows, self.general_skinny_rows)
        skinny = n <= skinny_rows and cfg.d_model % 64 == 0 and cfg.d_model <= 960 and (cfg.n_heads * cfg.head_dim) % 64 == 0
        mm = (lambda a, w, out: gemm_tn(a, w, out)) if skinny else (lambda a, w, out: torch.mm(a, w.t(), out=out))
        fold_mlp = not skinny and self.dtype != torch.float32 and cfg.d_ff % 8 == 0 and self.fold
        for l, W in enumerate(self.w.layers):
            if fused_attn is not None and self.fused_layer_ok(l, st):
                # decode rows of a 16-bit engine: the projection also forms the gate logits, and fused_attn(l) does the
                # post-processing, the cache append, the attention and its epilogue in one launch (writes buf zg)
                mm(xn, W["wqkv_ext"], b["qkvx"][:n])
                self._keep_projection(l, n)
                fused_attn(l)
            else:
                mm(xn, W["wqkv"], b["qkv"][:n])
                self._qkv_post(l, tok, pos, rows, last_pos, st, n)
                self._finish_attn(l, attn(l, b["q"][:n]))
            if skinny and "gu_il" in W:
                # the residual update rides on the output projection (h = resid_attn * x + post_attn * a) and the MLP's
                # pre-norm on the gate-up projection (a row scale of the product), whose epilogue is the SwiGLU
                gemm_tn(b["zg"][:n], W["wo"], b["h"][:n], epilogue=RESID, resid=x, ca=W["resid_attn"], cb=W["post_attn"])
                gemm_tn(b["h"][:n], W["gu_il"], b["act"][:n], epilogue=SWIGLU, norm_eps=self.eps)
            elif fold_mlp:
                # both residual updates are the library's C = alpha A B + beta C on the hidden in place and the MLP's pre-norm
                # is the row scale inside the SwiGLU launch; the block ends with the norm the next block reads
                torch.addmm(x, b["zg"][:n], W["wo"].t(), beta=W["resid_attn"], alpha=W["post_attn"], out=x)
                torch.mm(x, W["gu"].t(), out=b["gu"][:n])
                self._swiglu_norm(x, n)
                torch.addmm(x, b["act"][:n], W["down"].t(), beta=W["resid_mlp"], alpha=W["post_mlp"], out=x)
                if l + 1 < cfg.n_layers:
                    self._add_norm(x, x, 1.0, 0.0, n, None, b["xn"])
                continue
            else:
                mm(b["zg"][:n], W["wo"], b["a"][:n])
                # h = resid_attn * x + post_attn * a ; n = rmsnorm(h)
                self._add_norm(x, b["a"][:n], W["resid_attn"], W["post_attn"], n, b["h"], b["xn"])
                mm(xn, W["gu"], b["gu"][:n])
                self._swiglu(n)
            torch.mm(b["act"][:n], W["down"].t(), out=b["m"][:n])   # (K = d_ff: 26 K-steps per strip, the library is faster)
            # x = resid_mlp * h + post_mlp * m ; xn = rmsnorm(x) (next block's pre-norm, or the final norm)
            self._add_norm(b["h"][:n], b["m"][:n], W["resid_mlp"], W["post_mlp"], n, b["x"], b["xn"])
        return fold_mlp

    # ---- recorded passes
    def _planned(self, what: str, st: KVState, kind: str, n: int, values: dict, record) -> Tensor:
        """Run the pass that record() makes, from its recorded launch list: recorded the first time a pass of this
        shape class runs on the state (launched as it is recorded, so that a state's first pass waits for nothing), then only re-bound to
        the call's row counts and addresses (values).  The list is recorded again when an object it rests on is another one or
        elsewhere (weights and residual scalars, cache tensors, a switch of the launch plans)."""
        own_down = n <= self.skinny_rows or n >= self.big_rows or self.fold_down_rows[0] <= n <= self.fold_down_rows[1]
        key = (what, kind, n <= self.fold_qkv_rows, n <= self.fold_o_rows, n <= self.fold_gu_rows, own_down,
               self.fold_down_rows[0] <= n <= self.fold_down_rows[1], self._sums_ok(n), self.gemm_config, getattr(self.w, "scalar_epoch", 0))
        plans = self._plans.get(st)
        if plans is None:
            plans = self._plans[st] = {}
        plan = plans.get(key)
        if plan is None or not plan.guard.holds(self.w, st):
            if len(plans) >= 16:
                plans.clear()
            plan = PassPlan()
            plan.guard = Guard(self.w, st)
            self._rec = plan
            try:
                record()
            finally:
                self._rec = None
            plan.raw = self.hidden_is_raw
            plans[key] = plan.close()
        else:
            plan.run(values, L.stream_ptr(self.buf["x"]))
        self.hidden_is_raw = plan.raw
        return self.buf["x" if plan.raw else "xn"][:n]

    def _normed(self, rows: Tensor) -> Tensor:
        """The final norm of some rows of what _trunk returned, in place where it still has to be taken."""
        if self.hidden_is_raw and rows.size(0):
            self._add_norm(rows, rows, 1.0, 0.0, rows.size(0), None, rows)
        return rows

    def own_head_ok(self, n: int) -> bool:
        """Whether head_of runs the head GEMM of n rows on this library's kernel with the final norm in it: 16-bit engines up
        to head_own_rows rows.  Measured on UV-50M (32 768 x 640 head) as the time of a whole graph-replayed decode step
        against the vendor library's GEMM behind a norm launch: 0.3325 against 0.3338 ms at 192 rows, 0.3644 against 0.3699
        at 256, but 0.4137 against 0.4111 at 320 and 0.4363 against 0.4297 at 384 - so the switch sits at 288 rows.  (Alone,
        on cold weights, the kernel takes 11.5 - 25 us at 32 - 384 rows where the vendor library's takes 10 - 22 us plus ~6 us
        of norm launch; at 2048 rows 105 against 87 us.)"""
        cfg = self.cfg
        return (self.dtype in (torch.bfloat16, torch.float16) and n <= self.head_own_rows and cfg.d_model % 64 == 0
                and cfg.d_model >= 128 and cfg.vocab_size % 16 == 0)

    def head_of(self, hidden: Tensor) -> Tensor:
        """head() of what _trunk(defer_final_norm=True) returned: a raw hidden goes through this library's GEMM with the
        final norm as the row scale of the product (128 x 128 tiles; 256 x 256 where they fill the device in whole
        rounds), a normalised one through head()."""
        if not self.hidden_is_raw:
            return self.head(hidden)
        n = hidden.size(0)
        blocks = -(-n // 256)
        config = 5 if n > 384 and blocks % 2 == 0 else 6
        return gemm_tn(hidden, self.w.embed, norm_eps=self.eps, config=config)

    def head(self, hidden: Tensor) -> Tensor:
        """Raw tied-head output (n, V) in the activation dtype: the GEMM MathLM.logits runs before .float() and the
        softcap (model.py:824-827); the sampler applies the softcap."""
        return torch.mm(hidden, self.w.embed.t())

    def logits(self, hidden: Tensor) -> Tensor:
        """Softcapped fp32 logits of the normed hidden (MathLM.logits, model.py:824-827): on a 16-bit engine one GEMM whose
        epilogue rounds the product to the activation type and applies the softcap (the library's GEMM and the five
        elementwise passes over the (n, V) output took 130 us at 512 rows)."""
        a, bb, c = self.cfg.softcap
        W = self.w.embed
        if hidden.dim() == 2 and hidden.size(0) > 0 and self._own_logits_ok(hidden.dtype):
            hidden = hidden.contiguous()
            if gemm_supported(hidden, W, SOFTCAP):
                return gemm_tn(hidden, W, epilogue=SOFTCAP, ca=a, cb=bb, cap_c=c)
        return a * torch.sigmoid((self.head(hidden).float() + bb) / c)

    def _own_logits_ok(self, dtype: torch.dtype) -> bool:
        W = self.w.embed
        return dtype in (torch.bfloat16, torch.float16) and dtype == W.dtype and W.size(1) >= 128 and W.size(0) % 16 == 0

    def _raw_logits_ok(self, n: int, of: int | None = None) -> bool:
        """Whether _raw_logits takes n rows, of a hidden of `of` (n): what uvmi_head does, whose offsets into hidden and embedding are 32-bit."""
        W = self.w.embed
        of = n if of is None else of
        V, d = W.shape
        return (0 < n <= 1 << 16 and of <= 1 << 20 and self._own_logits_ok(self.dtype) and W.stride(1) == 1 and W.stride(0) % 8 == 0 and W.data_ptr() % 16 == 0
                and d % 64 == 0 and d <= 8192 and (V + 64) * W.stride(0) < 1 << 29 and (max(n, of) + 64) * d < 1 << 29)

    def _raw_logits(self, hidden: Tensor, rows: Tensor | None = None, advance: Tensor | None = None) -> Tensor:
        """logits() of rows `rows` (all) of what a trunk left un-normalised in buf x: the final norm is the row scale of the product, the rows are
        gathered by the GEMM's loads and positions `advance` counted up by its launch.  (One launch less a decode step, two
        less a prefill: a step of 37 rows 245.7 -> 242.1 us, of 512 413.5 -> 409.9, a prefill of 93 tokens, which waits for the host, 245 -> 241.  Of
        one row, where a head on 128-row tiles costs 2 us more with the norm in it and the host is as slow as the GPU, 188 -> 182 and 190 -> 181 on two machines,
        medians of 8 and 4 processes; from 1 to 384 rows no count is slower by more than the runs of one differ.)"""
        ca, cb, c = self.cfg.softcap
        W = self.w.embed
        n = hidden.size(0) if rows is None else rows.numel()
        out = torch.empty(n, W.size(0), dtype=torch.float32, device=hidden.device)
        g = gemm_args(hidden[:n], W, out, SOFTCAP, norm_eps=self.eps, ca=ca, cb=cb, cap_c=c)
        h = L.HeadArgs(C.addressof(g), None if rows is None else rows.data_ptr(), hidden.size(0), None if advance is None else advance.data_ptr(),
                       0 if advance is None else advance.numel())
        L.check(L.lib().uvmi_head(C.byref(h), L.stream_ptr(out)), "uvmi_head")
        return out

    # ------------------------------------------------------------------------------------------------ decode
    @torch.no_grad()
    def decode_step(self, tok: Tensor, st: KVState, num_splits: dict | None = None, fuse: bool = True) -> Tensor:
        """One token for all B rows at per-row st.pos (reference: decode_step_fast, fast_decode.py:272-334): append K/V
        at pos first, attend lo..pos, then st.pos += 1.  Returns the final normed hidden (B, d)."""
        return self._decode(tok, st, num_splits, fuse, False)

    @torch.no_grad()
    def decode_logits(self, tok: Tensor, st: KVState, num_splits: dict | None = None) -> Tensor:
        """logits(decode_step(tok, st, num_splits)); where the step's plan leaves the hidden as it is, the head takes the final norm."""
        return self._decode(tok, st, num_splits, True, True)

    def _decode(self, tok: Tensor, st: KVState, num_splits: dict | None, fuse: bool, head: bool) -> Tensor:
        cfg = self.cfg
        B = tok.numel()
        pos, starts = st.pos, st.starts
        ns = num_splits or {}
        fused = None
        if self.fuse_qkv and not num_splits and fuse:
            fused = lambda l, oproj=False: self.fused_cache_attention(l, tok, st, pos, starts, B, oproj=oproj)
            kind = self._pass_kind(B, True, st)
            if kind in ("lean", "lean-o", "folded") and self.qkvx_keep is None:
                assert B <= self.max_tokens and B <= st.B
                # (a recorded list takes addresses only, so what its launches assume of the arrays is checked on every call)
                assert all(t.dtype == torch.int64 and t.is_contiguous() and t.numel() >= B for t in (tok, pos, starts))
                whole = B == pos.numel()     # (a step of fewer rows than the state has still moves every position)
                if head and self._raw_logits_ok(B):
                    h = self._planned("decode-raw", st, kind, B, dict(n=B, tok=tok.data_ptr(), pos=pos.data_ptr(), starts=starts.data_ptr()),
                                      lambda: self._trunk(tok, pos, B, None, st=st, fused_attn=fused, final_norm=False))
                    return self._raw_logits(h, advance=pos)
                h = self._planned("decode" if whole else "decode-part", st, kind, B,
                                  dict(n=B, tok=tok.data_ptr(), pos=pos.data_ptr(), starts=starts.data_ptr()),
                                  lambda: self._trunk(tok, pos, B, None, st=st, fused_attn=fused, advance=whole))
                if not whole:
                    st.pos.add_(1)
                return self.logits(h) if head else h

        def attn(l, q):
            key = "global" if cfg.is_global(l) else "local"
            if ns.get(key) in (None, 1):
                return self.cache_attention(l, q, st, pos, starts, B)
            glob = cfg.is_global(l)
            k, v, ks, vs = st.cache(l)
            return decode_attention(q, k, v, pos, starts, cfg.attn_scale, window=st.window(l), ring=not glob,
                                    k_scale=ks, v_scale=vs, num_splits=ns[key])

        h = self._trunk(tok, pos, B, attn, st=st, fused_attn=fused)
        st.pos.add_(1)
        return self.logits(h) if head else h

    # ------------------------------------------------------------------------------------------------ prefill
    def _staging(self, n: int):
        """n int64 of pinned host memory out of a small ring, and the event to record behind the launch that reads it: a buffer
        is handed out again, or given back to the allocator, only after that launch."""
        self._stage_at = (self._stage_at + 1) % len(self._stage)
        st = self._stage[self._stage_at]
        st.wait()
        if st.buf is None or st.buf.numel() < n:
            st.buf, st.event = torch.empty(max(1024, n + n // 4), dtype=torch.int64, pin_memory=True), torch.cuda.Event()
        return st.buf, st.event

    def _pack(self, prompts, rows, max_len: int, left_pad: bool, st: KVState | None = None, idx: Tensor | None = None, lens=None,
              check: Tensor | None = None, check_zero: bool = False) -> dict:
        """pack_prompts; st: also bind its rows to the prompts; idx (n, T) with lens instead of prompts: right-aligned prompts
        already on the device; check: n int64 of the device that the caller wants to see: pk["check"]() waits for this launch
        and gives them; check_zero: prompts whose entry is not zero leave the state as it is.  The launch reads the host's tables in pinned memory: a copy to the device would make the host wait
        for the passes still running (pageable memory) or cost the GPU 20 us (pinned memory)."""
        if idx is None:
            lens = np.fromiter((len(p) for p in prompts), dtype=np.int64, count=len(prompts))
        n = len(lens)
        assert lens.min() > 0
        T = int(lens.max())
        assert T <= max_len
        N = int(lens.sum())
        assert N <= self.max_tokens, f"{N} prefill tokens exceed the engine's max_tokens {self.max_tokens}"
        rows_np = np.asarray(rows, dtype=np.int64)
        assert len(rows_np) == n
        n_tok = N if idx is None else 0
        buf, ev = self._staging(4 * n + 1 + n_tok)
        h = buf.numpy()
        h[0] = 0
        np.cumsum(lens, out=h[1:n + 1])
        h[n + 1:2 * n + 1] = rows_np
        h[2 * n + 1:3 * n + 1] = (T - lens) if left_pad else 0
        if idx is None:
            np.concatenate([np.asarray(p, dtype=np.int64) for p in prompts], out=h[4 * n + 1:4 * n + 1 + N])   # (prompts may be lists or int arrays)
        pinned = n <= 2047
        host = buf if pinned else buf[:4 * n + 1 + n_tok].to(self.device)
        src = host.data_ptr()
        out = torch.empty(4 * N + 5 * n + 1, dtype=torch.int64, device=self.device)
        tok, pos, row, last, last_idx, cu_t, rows_t, starts_t, ends = out.split([N, N, N, N, n, n + 1, n, n, n])
        pk = dict(N=N, tok=tok, pos=pos, row=row, last=last, cu=cu_t, last_idx=last_idx, rows=rows_t, starts=starts_t, ends=ends,
                  rows_h=(int(rows_np.min()), int(rows_np.max())))
        at = out.data_ptr()
        a = L.PromptTablesArgs(n=n, n_tokens=N, idx_ld=0 if idx is None else idx.size(1), cu=src, row=src + 8 * (n + 1), start=src + 8 * (2 * n + 1),
                               tok=src + 8 * (4 * n + 1) if idx is None else idx.data_ptr(), tok_t=at, pos_t=at + 8 * N, row_t=at + 16 * N, last_t=at + 24 * N,
                               last_idx=at + 32 * N, cu_out=cu_t.data_ptr(), row_out=rows_t.data_ptr(), start_out=starts_t.data_ptr(), end_out=ends.data_ptr())
        if st is not None:
            self._check_rows(pk, st)
            a.st_pos, a.st_starts = st.pos.data_ptr(), st.starts.data_ptr()
        if check is not None:
            assert pinned and check.dtype == torch.int64 and check.is_contiguous() and check.numel() == n
            a.check_in, a.check_out, a.check_zero = check.data_ptr(), src + 8 * (3 * n + 1), int(check_zero)

            def seen():
                ev.synchronize()
                return h[3 * n + 1:4 * n + 1].copy()
            pk["check"] = seen
        L.check(L.lib().uvmi_prompt_tables(C.byref(a), L.stream_ptr(out)), "uvmi_prompt_tables")
        ev.record(torch.cuda.current_stream(self.device))
        return pk

    @staticmethod
    def _check_rows(pk: dict, st: KVState):
        if pk["rows_h"][0] < 0 or pk["rows_h"][1] >= st.pos.numel():
            raise IndexError(f"cache rows {pk['rows_h'][0]}..{pk['rows_h'][1]} of a state with {st.pos.numel()} rows")

    def pack_prompts(self, prompts: list[list[int]], rows: list[int], max_len: int, left_pad: bool = True) -> dict:
        """Packed indices of a prefill call (reference: prefill_packed_host, fast_decode.py:210-269): per packed token its id,
        position, cache row and the last position of its prompt; cu_seqlens; the packed index of every prompt's last token; per
        prompt the cache row, start and end position.  All as device tensors: the host uploads the tokens and one line
        per prompt, a launch forms the per-token tables."""
        return self._pack(prompts, rows, max_len, left_pad)

    @staticmethod
    def bind_prompts(pk: dict, st: KVState):
        """Point the cache rows of a packed prefill at their prompts: starts = first position, pos = next position."""
        st.starts[pk["rows"]] = pk["starts"]
        st.pos[pk["rows"]] = pk["ends"]

    @torch.no_grad()
    def mixed_step(self, pk: dict, tok_d: Tensor, pos_d: Tensor, starts_d: Tensor, rows_d: Tensor, st: KVState) -> tuple[Tensor, Tensor]:
        """One forward pass over a mixed batch: the packed prompts of `pk` (prefilled into their cache rows) followed by
        n_d decode rows (token tok_d at position pos_d of cache row rows_d; rows_d < 0 marks padding).  Every GEMM, norm
        and the fused QKV post-processing / cache append run once over all N_p + n_d token rows; attention runs as one
        packed causal launch over the prompt tokens and one cache launch over the decode rows per layer.  The reference
        runs these as two passes (its refill prefill, then the decode step: model.py:1296-1313, 1321-1330).
        Returns the final normed hidden of each prompt's last token and of each decode row.  Does not advance st.pos of
        the decode rows (the caller's slot table does), but binds the prompts' rows."""
        Np, nd = pk["N"], tok_d.numel()
        N = Np + nd
        tables = torch.empty(4, N, dtype=torch.int64, device=self.device)
        tok, pos, rows, last = tables.unbind(0)
        tok_d, pos_d, rows_d = (t.to(torch.int64).contiguous() for t in (tok_d, pos_d, rows_d))
        self._check_rows(pk, st)
        a = L.PromptTablesArgs(n=pk["rows"].numel(), n_tokens=Np, nd=nd, cu=pk["cu"].data_ptr(), row=pk["rows"].data_ptr(), start=pk["starts"].data_ptr(),
                               tok=pk["tok"].data_ptr(), tok_d=tok_d.data_ptr(), pos_d=pos_d.data_ptr(), rows_d=rows_d.data_ptr(), tok_t=tok.data_ptr(),
                               pos_t=pos.data_ptr(), row_t=rows.data_ptr(), last_t=last.data_ptr())
        L.check(L.lib().uvmi_prompt_tables(C.byref(a), L.stream_ptr(tables)), "uvmi_prompt_tables")
        h = self.mixed_trunk(tok, pos, rows, last, Np, nd, pk["cu"], starts_d, st, final_norm=False)
        b = L.PromptTablesArgs(n=a.n, cu=a.cu, row=a.row, start=a.start, st_pos=st.pos.data_ptr(), st_starts=st.starts.data_ptr())
        L.check(L.lib().uvmi_prompt_tables(C.byref(b), L.stream_ptr(tables)), "uvmi_prompt_tables")   # (after the pass: pos_d may be a view of st.pos)
        return self._normed(h.index_select(0, pk["last_idx"])), self._normed(h[Np:N])

    def mixed_trunk(self, tok: Tensor, pos: Tensor, rows: Tensor, last: Tensor, Np: int, nd: int, cu: Tensor, starts_d: Tensor,
                    st: KVState, final_norm: bool = True) -> Tensor:
        """The pass of mixed_step over already concatenated per-token arrays (Np packed prompt tokens, then nd decode rows;
        cu: the prompts' cu_seqlens on the device).  Allocation-free apart from the packed attention output, so a caller
        that builds the arrays on the device can capture it in a graph.  Returns the final normed hidden (Np + nd, d); final_norm
        False: as in _trunk."""
        cfg, b = self.cfg, self.buf
        N = Np + nd
        assert N <= self.max_tokens, f"{N} token rows exceed the engine's max_tokens {self.max_tokens}"
        pos_d, rows_d = pos[Np:N], rows[Np:N]

        def attn(l, q):
            return [(0, self.prompt_attention(l, q[:Np], Np, cu)),
                    (Np, self.cache_attention(l, q[Np:N], st, pos_d, starts_d, nd, rows=rows_d, off=Np))]

        run = lambda: self._trunk(tok[:N], pos[:N], N, attn, rows=rows[:N], last_pos=last[:N], st=st, final_norm=final_norm)
        if (Np > 0 and nd > 0 and self._pass_kind(N, False, st) == "packed" and self.prompt_attention_plannable() and self._append_fused(st)
                and all(self.cache_attention_plannable(l, st) for l in range(cfg.n_layers))):
            assert all(t.dtype == torch.int64 and t.stride(0) == 1 for t in (tok, pos, rows, last, starts_d))
            at = lambda name: b[name].data_ptr() + Np * b[name].stride(0) * b[name].element_size()
            values = dict(n=N, Np=Np, nd=nd, tok=tok.data_ptr(), pos=pos.data_ptr(), rows=rows.data_ptr(), last=last.data_ptr(), cu=cu.data_ptr(),
                          n_seg=cu.numel() - 1, pos_d=pos_d.data_ptr(), rows_d=rows_d.data_ptr(), starts_d=starts_d.data_ptr(),
                          q_d=at("q"), vhat_d=at("vhat"), gate_d=at("gate"), zg_d=at("zg"))
            return self._planned("mixed" if final_norm else "mixed-raw", st, "packed", N, values, run)
        return run()

    @torch.no_grad()
    def prefill(self, prompts: list[list[int]], rows: list[int], st: KVState, left_pad: bool = True) -> Tensor:
        """Packed prefill of whole prompts into cache rows `rows` (reference: prefill_packed_host, fast_decode.py:210-269):
        the real tokens of all prompts run back to back through the trunk with causal (and, on local layers, windowed)
        attention over their own unquantized K/V; only the cache write quantises.  left_pad keeps the reference's
        positions (token j of a prompt of length n sits at T - n + j, T = longest prompt of the call) so the cache
        layout equals the reference's; left_pad=False starts every prompt at position 0.  Sets st.pos / st.starts of the
        rows and returns the final normed hidden of each prompt's last token (len(prompts), d)."""
        return self._prefill(self._pack(prompts, rows, st.max_len, left_pad, st), st)

    @torch.no_grad()
    def prefill_logits(self, prompts: list[list[int]], rows: list[int], st: KVState, left_pad: bool = True) -> Tensor:
        """logits(prefill(prompts, rows, st, left_pad)), without the launches that gather and norm the prompts' last rows."""
        return self._prefill(self._pack(prompts, rows, st.max_len, left_pad, st), st, True)

    @torch.no_grad()
    def prefill_matrix(self, idx: Tensor, lens, rows, st: KVState, check: Tensor | None = None):
        """prefill(left_pad=True) of the prompts that stand right-aligned in idx (n, T), an int64 matrix on the engine's device: the
        last lens[a] (host) tokens of row a.  The token ids never visit the host.  check: n int64 of the device that have to be
        zero; also returns a function that gives them without waiting for the pass.  A prompt whose entry is not zero leaves
        the state as it is - cache row, pos and starts -, so the caller may raise when it sees that."""
        return self._prefill_matrix(idx, lens, rows, st, check, False)

    @torch.no_grad()
    def prefill_matrix_logits(self, idx: Tensor, lens, rows, st: KVState, check: Tensor | None = None):
        """prefill_matrix with the logits of the prompts' last rows in place of their hidden."""
        return self._prefill_matrix(idx, lens, rows, st, check, True)

    def _prefill_matrix(self, idx: Tensor, lens, rows, st: KVState, check: Tensor | None, head: bool):
        assert idx.dtype == torch.int64 and idx.is_contiguous() and idx.size(0) == len(lens) and idx.size(1) >= int(lens.max())
        pk = self._pack(None, rows, st.max_len, True, st, idx, lens, check, check_zero=check is not None)
        h = self._prefill(pk, st, head)
        return h if check is None else (h, pk["check"])

    def _prefill(self, pk: dict, st: KVState, head: bool = False) -> Tensor:
        N = pk["N"]

        def attn(l, q, gemm=None):
            return self.prompt_attention(l, q, N, pk["cu"], gemm)

        tok, pos, row, last, cu = pk["tok"], pk["pos"], pk["row"], pk["last"], pk["cu"]
        run = lambda: self._trunk(tok, pos, N, attn, rows=row, last_pos=last, st=st, final_norm=False, oproj=self.prompt_attention_plannable())
        if self._pass_kind(N, False, st) == "packed" and self.prompt_attention_plannable() and self._append_fused(st):
            h = self._planned("prefill", st, "packed", N, dict(n=N, Np=N, tok=tok.data_ptr(), pos=pos.data_ptr(), rows=row.data_ptr(), last=last.data_ptr(),
                                                                cu=cu.data_ptr(), n_seg=cu.numel() - 1), run)
        else:
            h = run()
        if head and self.hidden_is_raw and self._raw_logits_ok(pk["last_idx"].numel(), h.size(0)):
            return self._raw_logits(h, rows=pk["last_idx"])
        h = self._normed(h.index_select(0, pk["last_idx"]))   # (the norm of the prompts' last rows only)
        return self.logits(h) if head else h

    # ------------------------------------------------------------------------------------------------ generation
    @torch.no_grad()
    def generate(self, prompts: list[list[int]], max_new: int, temperature: float = 0.0, seed: int = 0,
                 max_len: int | None = None, use_graph: bool = False, return_logp: bool = False, top_k: int = 0,
                 top_p: float = 1.0, kv_dtype: str = "int8"):
        """Static-batch generation (reference: generate, model.py:1228-1263): packed prefill of all prompts, then
        lockstep decode.  temperature <= 0: greedy.  Otherwise the fused sampler with Philox uniforms keyed by
        (seed, request = prompt index, token index), truncated by top_k / top_p as sample() does (model.py:1200-1209)."""
        cfg, dev = self.cfg, self.device
        B = len(prompts)
        T = max(len(p) for p in prompts)
        st = KVState(cfg, B, max_len or (T + max_new), dev, kv_dtype=kv_dtype, dtype=self.dtype)
        req = torch.arange(B, dtype=torch.long, device=dev)
        ti = torch.zeros(B, dtype=torch.long, device=dev)

        def draw(hidden):
            xh = self.head(hidden)
            if temperature <= 0:
                return greedy_sample(xh, cfg.softcap)
            return fused_sample_seeded(xh, seed, req, ti, cfg.softcap, temperature, top_k=top_k, top_p=top_p)

        tok, lp = draw(self.prefill(prompts, list(range(B)), st))
        toks, lps = [tok.clone()], [lp.clone()]
        cur = tok.clone()
        graph = None

        def step():
            ti.add_(1)
            t, l_ = draw(self.decode_step(cur, st))
            cur.copy_(t)
            lpbuf.copy_(l_)

        lpbuf = torch.zeros(B, dtype=torch.float32, device=dev)
        for i in range(max_new - 1):
            if use_graph:
                if graph is None:
                    pos0, ti0, cur0 = st.pos.clone(), ti.clone(), cur.clone()
                    s = torch.cuda.Stream()
                    s.wait_stream(torch.cuda.current_stream())
                    with torch.cuda.stream(s):
                        step()
                    torch.cuda.current_stream().wait_stream(s)
                    st.pos.copy_(pos0); ti.copy_(ti0); cur.copy_(cur0)
                    graph = torch.cuda.CUDAGraph()
                    with torch.cuda.graph(graph):
                        step()
                    st.pos.copy_(pos0); ti.copy_(ti0); cur.copy_(cur0)
                graph.replay()
            else:
                step()
            toks.append(cur.clone())
            lps.append(lpbuf.clone())
        out = torch.stack(toks, 1).tolist()
        if return_logp:
            return out, torch.stack(lps, 1).cpu().numpy()
        return out
