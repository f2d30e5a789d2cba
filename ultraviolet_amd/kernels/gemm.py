"""Skinny 16-bit GEMM of a small decode step's projections (uvmi_gemm_tn): out = a @ w.T with fp32 accumulation,
optionally with the SwiGLU of the MLP folded into the epilogue.  Stands in for the F.linear calls of the reference's
fused inference path (ultraviolet/model.py:302-335, 388-391) when the batch is a few hundred rows."""
from __future__ import annotations

import ctypes as C

import torch
from torch import Tensor

from .. import _lib as L

STORE, SWIGLU, RESID, SOFTCAP = 0, 1, 2, 4


def gemm_supported(a: Tensor, w: Tensor, epilogue: int = STORE) -> bool:
    if not (a.is_cuda and a.dim() == 2 and w.dim() == 2 and a.dtype == w.dtype and a.dtype in (torch.float16, torch.bfloat16)):
        return False
    if a.stride(1) != 1 or w.stride(1) != 1 or a.size(1) != w.size(1) or a.data_ptr() % 16 or w.data_ptr() % 16:
        return False
    n_out = w.size(0) // 2 if epilogue == SWIGLU else w.size(0)
    return bool(L.lib().uvmi_gemm_tn_supported(L.dtype_code(a.dtype), a.size(0), w.size(0), a.size(1), a.stride(0), w.stride(0),
                                               n_out, epilogue))


def gemm_args(a: Tensor, w: Tensor, out: Tensor, epilogue: int = STORE, *, norm_eps: float | None = None, resid: Tensor | None = None,
              ca: float = 1.0, cb: float = 1.0, cap_c: float = 0.0, config: int = 0):
    """The uvmi_gemm_args block of gemm_tn."""
    M, K = a.shape
    N = w.size(0)
    assert out.shape == (M, N // 2 if epilogue == SWIGLU else N) and out.dtype == (torch.float32 if epilogue == SOFTCAP else a.dtype)
    assert out.stride(1) == 1 and a.stride(1) == 1 and w.stride(1) == 1
    rp, ldr = None, 0
    if epilogue == RESID:
        assert resid is not None and resid.shape == (M, N) and resid.dtype == a.dtype and resid.stride(1) == 1
        rp, ldr = resid.data_ptr(), resid.stride(0)
    return L.GemmArgs(a.data_ptr(), w.data_ptr(), out.data_ptr(), L.dtype_code(a.dtype), M, N, K, a.stride(0), w.stride(0), out.stride(0),
                      epilogue, norm_eps is not None, norm_eps or 0.0, rp, ldr, ca, cb, config, cap_c)


TILED, STREAM, BIG = range(3)   # UVMI_GEMM_PATH_*


def gemm_path(g) -> tuple[int, int, int]:
    """Which kernel takes a gemm_args block (TILED, STREAM or BIG), and its tile's rows and columns."""
    rows, cols = C.c_int(), C.c_int()
    kind = L.lib().uvmi_gemm_tn_path(C.byref(g), C.byref(rows), C.byref(cols))
    if kind < 0:
        L.check(kind, "uvmi_gemm_tn")
    return kind, rows.value, cols.value


def gemm_tn(a: Tensor, w: Tensor, out: Tensor | None = None, epilogue: int = STORE, *, norm_eps: float | None = None,
            resid: Tensor | None = None, ca: float = 1.0, cb: float = 1.0, cap_c: float = 0.0, config: int = 0) -> Tensor:
    """a (M, K) @ w (N, K).T -> (M, N); with epilogue=SWIGLU w is interleave_gate_up(w_gate, w_up) and the result is
    silu(a @ w_gate.T) * (a @ w_up.T), (M, N / 2); with epilogue=RESID the result is ca * resid + cb * (a @ w.T) (the
    block's residual update, ultraviolet/model.py:567-571); with epilogue=SOFTCAP it is ca * sigmoid((x + cb) / cap_c) in fp32
    of the rounded product x (the logits, model.py:824-827).  norm_eps: a stands for rmsnorm(a) with that epsilon (the
    pre-norm of the block folded into the projection as a row scale of the product).  Raises UvmiError for shapes the
    kernel does not take.  config (tuning / tests): 0 built-in choice, else a form of the kernel (uvmi_gemm_args.config)."""
    if out is None:
        out = torch.empty(a.size(0), w.size(0) // 2 if epilogue == SWIGLU else w.size(0), dtype=torch.float32 if epilogue == SOFTCAP else a.dtype, device=a.device)
    g = gemm_args(a, w, out, epilogue, norm_eps=norm_eps, resid=resid, ca=ca, cb=cb, cap_c=cap_c, config=config)
    L.check(L.lib().uvmi_gemm_tn_ex(C.byref(g), L.stream_ptr(a)), "uvmi_gemm_tn")
    return out


def interleave_gate_up(w_gate: Tensor, w_up: Tensor) -> Tensor:
    """(f, K), (f, K) -> (2 f, K) in slabs of 16 rows [gate 0..15 | up 0..15 | gate 16..31 | ...]: the weight layout of the
    SWIGLU epilogue (f % 16 == 0)."""
    f, K = w_gate.shape
    assert w_up.shape == (f, K) and f % 16 == 0
    return torch.stack([w_gate.view(f // 16, 16, K), w_up.view(f // 16, 16, K)], 1).reshape(2 * f, K).contiguous()
