"""The launch list of a forward pass, prepared once and issued with one native call per pass (uvmi_run_ops).

A pass is ~50 launches whose arguments are the same from call to call except for the number of token rows and the addresses
of the per-call arrays.  Preparing them one by one from Python costs ~12 us each, twice what the GPU needs for the launch
on a small batch; a prepared list costs ~3 us a launch.  A list holds argument blocks (addresses and sizes), never
results: every launch runs on every call."""
from __future__ import annotations

import ctypes as C
from itertools import chain
from operator import is_

import torch
from torch import Tensor

from .. import _lib as L


class Guard:
    """The objects that recorded launches took addresses and numbers from - weights, residual scalars, cache tensors - and where the
    tensors among them were: one may be replaced, or keep its object and move (`.data = `).  Every pass asks, so it is two walks in C
    over ~170 objects (10 us; the launches of one layer take 15)."""

    _END = object()

    def __init__(self, weights, state):
        self.objects = tuple(self._of(weights, state))
        live = {id(W[k]) for W in weights.layers for k in ("wqkv", "gu") if k in W}   # (no launch of this library in a list reads these)
        self.tensors = [t for t in self.objects if isinstance(t, Tensor) and id(t) not in live]
        self.at = list(map(Tensor.data_ptr, self.tensors))
        self.every = list(range(len(self.tensors)))

    def _of(self, w, st):
        return chain((w.embed, w.value_embed, w.inv_freq), *map(dict.values, w.layers), st.k, st.v, st.k_scale, st.v_scale, (self._END,))

    def holds(self, weights, state) -> bool:
        return all(map(is_, self.objects, self._of(weights, state))) and _same_addresses(self.tensors, self.at, self.every)


# (what torch's graph trees compare their static inputs with: half the time of a list of data_ptr() calls)
_same_addresses = getattr(torch._C, "_tensors_data_ptrs_at_indices_equal", None) or (lambda ts, at, _: list(map(Tensor.data_ptr, ts)) == at)


class PassPlan:
    def __init__(self):
        self.items = []     # ("ops", [(kind, args struct)]) or ("call", function of the pass's values), in launch order
        self.keep = []      # what the argument blocks point into
        self.fields = {}    # name of a per-call value -> [(struct, field)] that hold it
        self.bound = {}     # the values they hold now
        self.guard = None   # Guard of what the recorded arguments were taken from

    def op(self, kind: int, args, keep=(), **per_call):
        """A launch; per_call: field of args (or (struct, field)) = name of the per-call value it holds."""
        if not self.items or self.items[-1][0] != "ops":
            self.items.append(("ops", []))
        self.items[-1][1].append((kind, args))
        self.keep.append((args, keep))
        for field, name in per_call.items():
            self.field(args, field, name)

    def field(self, struct, field: str, name: str):
        self.fields.setdefault(name, []).append((struct, field))

    def call(self, fn):
        """Work between the launches that is not this library's (a GEMM of the vendor library)."""
        self.items.append(("call", fn))

    def close(self):
        self.segments = []
        for what, item in self.items:
            if what == "ops":
                kinds = (C.c_int * len(item))(*[k for k, _ in item])
                args = (C.c_void_p * len(item))(*[C.addressof(a) for _, a in item])
                item = (kinds, args, len(item))
            self.segments.append((what, item))
        return self

    def run(self, values: dict, stream: int):
        """values: the pass's row counts and addresses by name; only the fields of values that changed are rewritten."""
        for name, v in values.items():
            if self.bound.get(name, self) != v:
                self.bound[name] = v
                for s, f in self.fields.get(name, ()):
                    setattr(s, f, v)
        run_ops = L.lib().uvmi_run_ops
        for what, item in self.segments:
            if what == "ops":
                rc = run_ops(*item, stream)
                if rc:
                    L.check(rc, "uvmi_run_ops")
            else:
                item(values)


_ENTRY = {L.OP_GEMM: "uvmi_gemm_tn_ex", L.OP_DECODE_ATTN: "uvmi_decode_attn", L.OP_QKV_POST: "uvmi_qkv_post", L.OP_PREFILL_ATTN: "uvmi_prefill_attn",
          L.OP_QKV_PROJ: "uvmi_qkv_proj", L.OP_PREFILL_ATTN_O: "uvmi_prefill_attn_o", L.OP_GEMM_RESID: "uvmi_gemm_resid",
          L.OP_GEMM_SUMS: "uvmi_gemm_sums"}


def launch(kind: int, args, stream: int):
    """One operation at once."""
    if kind in _ENTRY:
        L.check(getattr(L.lib(), _ENTRY[kind])(C.byref(args), stream), _ENTRY[kind])
    else:
        L.check(L.lib().uvmi_run_ops((C.c_int * 1)(kind), (C.c_void_p * 1)(C.addressof(args)), 1, stream), "uvmi_run_ops")
