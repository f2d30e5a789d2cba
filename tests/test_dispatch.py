"""Which calls of decode_attention may launch past the dispatcher: those that no transform, mode, tracer or gradient sees.
No GPU: the launch and the registered op are replaced by recorders."""
import ctypes
import subprocess

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from ultraviolet_amd.kernels import decode_attn as D


class _Passing(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Subclass(torch.Tensor):
    pass


@pytest.fixture
def route(monkeypatch):
    """call(q, k, v) -> "launch" or "op"."""
    taken = []
    monkeypatch.setattr(D.L, "require_cuda", lambda *t: None)
    monkeypatch.setattr(D, "_launch", lambda q, *a, **k: taken.append("launch") or torch.zeros_like(q))
    monkeypatch.setattr(D, "_decode_attn_op", lambda q, *a, **k: taken.append("op") or torch.zeros_like(q))
    idx = torch.zeros(2, dtype=torch.long)

    def call(q, k, v):
        D.decode_attention(q, k, v, idx, idx, 0.1, num_splits=1)
        return taken.pop()
    return call


def _qkv():
    return torch.randn(2, 8, 64).half(), torch.randn(2, 1, 32, 64).half(), torch.randn(2, 1, 32, 64).half()


def test_plain_call_launches(route):
    assert route(*_qkv()) == "launch"


@pytest.mark.parametrize("which", [0, 1, 2])
def test_gradient_and_subclass_of_any_operand_reach_the_op(route, which):
    t = list(_qkv())
    t[which] = t[which].clone().requires_grad_()
    assert route(*t) == "op"
    t = list(_qkv())
    t[which] = t[which].as_subclass(_Subclass)
    assert route(*t) == "op"


def test_modes_and_transforms_reach_the_op(route):
    with _Passing():
        assert route(*_qkv()) == "op"
    with torch.autograd.forward_ad.dual_level():
        assert route(*_qkv()) == "op"
    seen = []
    q, k, v = _qkv()
    torch.func.vmap(lambda a: (seen.append(route(a, k, v)), a)[1])(q[None])
    assert seen == ["op"]


@pytest.mark.parametrize("q_dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kv_dtype", [torch.int8, torch.float16, torch.bfloat16])
def test_splits_of_a_call_that_names_none(monkeypatch, q_dtype, kv_dtype):
    """The native call and the general path cut a row alike, and never into chunks beyond one per compute unit or under 128 keys where the
    matrix-core kernel serves; the generic kernel's geometries are cut as default_splits has it."""
    monkeypatch.setattr(D, "_device_cus", lambda index: 256)
    native = D.L.lib().uvmi_decode_attn_splits
    for G, hd, S, ring in [(8, 64, 4096, False), (8, 64, 4098, False), (1, 64, 31, False), (4, 64, 250, True), (4, 64, 256, True), (9, 64, 4096, False), (8, 128, 4096, False)]:
        for n in (0, 1, 3, 32, 64, 65, 128, 129, 256, 257, 5000):
            for ctx in (0, 1, 127, 800, 1023, 1024, 2048, 2400, 4096, 100000):
                s = D._own_splits(q_dtype, kv_dtype, n, G, hd, S, ring, ctx, torch.device("cuda", 0))
                assert s == native(D.L.dtype_code(q_dtype), D.L.dtype_code(kv_dtype), n, G, hd, S, ring, ctx, 256)
                if hd == 128 or G == 9 or S == 31 or q_dtype == torch.float32:
                    assert s == D.default_splits(n, ctx, torch.device("cuda", 0))
                elif s > 1 and S % 32 == 0 and kv_dtype in (torch.int8, q_dtype):
                    assert s * n <= 256 and ctx // s >= 128


def _cache(kv_dtype, S, pitch, at=0, KH=1):
    """(2, KH, S, 64) with rows `pitch` elements apart from element `at` on."""
    return torch.zeros(at + 2 * KH * S * pitch, dtype=kv_dtype)[at:].view(2, KH, S, pitch)[..., :64]


@pytest.mark.parametrize("kv_dtype,S,pitch,k_at,v_at,s_at,q_at,scale,ring", [
    (torch.int8, 2048, 64, 0, 0, 0, 0, 0.1, False), (torch.int8, 2048, 72, 0, 0, 0, 0, 0.1, False), (torch.int8, 2048, 80, 0, 0, 0, 0, 0.1, False),
    (torch.int8, 2048, 64, 8, 0, 0, 0, 0.1, False), (torch.int8, 2048, 64, 16, 4, 4, 8, 0.1, False), (torch.int8, 2048, 64, 0, 2, 0, 0, 0.1, False),
    (torch.int8, 2048, 64, 0, 0, 2, 0, 0.1, False), (torch.int8, 2048, 64, 0, 0, 0, 4, 0.1, False), (torch.int8, 2048, 64, 0, 0, 0, 0, -0.1, False),
    (torch.int8, 2048, 64, 0, 0, 0, 0, 0.0, False), (torch.int8, 2048, 64, 0, 0, 0, 0, 0.1, True), (torch.int8, 2052, 64, 0, 0, 0, 0, 0.1, True),
    (torch.float16, 2048, 64, 0, 0, 0, 0, 0.1, False), (torch.float16, 2048, 68, 0, 0, 0, 0, 0.1, False), (torch.float16, 2048, 72, 8, 4, 0, 8, 0.1, False),
    (torch.float16, 2048, 64, 4, 0, 0, 0, 0.1, False), (torch.float16, 2048, 64, 0, 2, 0, 0, 0.1, False), (torch.bfloat16, 2048, 64, 0, 0, 0, 0, 0.1, False)])
def test_splits_of_a_call_follow_the_kernel_that_serves_it(monkeypatch, kv_dtype, S, pitch, k_at, v_at, s_at, q_at, scale, ring):
    """Strides and addresses that the matrix-core kernel does not take leave a call to the generic one, whose rows are cut by default_splits: in eager
    calls by uvmi_decode_attn_path's answer, in traced ones by the same rules over strides and offsets."""
    taken = []
    monkeypatch.setattr(D, "_device_cus", lambda index: 256)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(D.L, "require_cuda", lambda *t: None)
    monkeypatch.setattr(D, "_launch", lambda q, *a, **k: taken.append(a[9]) or torch.zeros_like(q))
    monkeypatch.setattr(D, "_decode_attn_op", lambda q, *a, **k: taken.append(a[9]) or torch.zeros_like(q))
    q = torch.zeros(q_at + 2 * 8 * 64, dtype=torch.float16)[q_at:].view(2, 8, 64)
    k, v = _cache(kv_dtype, S, pitch, k_at), _cache(kv_dtype, S, pitch, v_at)
    ks, vs = (torch.zeros(s_at + 2 * S, dtype=torch.float16)[s_at:].view(2, 1, S) for _ in range(2)) if kv_dtype == torch.int8 else (None, None)
    pos = torch.zeros(2, dtype=torch.long)
    a, keep = D.build_attn_args(q, k, v, pos, pos, scale, 0, ring, ks, vs, 1, torch.zeros_like(q))
    path = D.L.lib().uvmi_decode_attn_path
    monkeypatch.setattr(path, "argtypes", [ctypes.POINTER(D.L.AttnArgs)])   # (another test binds the library to a structure of its own)
    served = path(ctypes.byref(a))
    splits = lambda: D.decode_attention(q, k, v, pos, pos, scale, ring=ring, k_scale=ks, v_scale=vs)
    splits()
    with _Passing():
        splits()
    want = D._own_splits(q.dtype, kv_dtype, 2, 8, 64, S, ring, S) if served == 1 else D.default_splits(2, S)
    assert served in (0, 1) and taken == [want] * 2 and (served == 1 or want == 8)


def test_rows_that_default_splits_leaves_whole_are_whole_by_either_rule():
    """What the native call rests on: it asks for the kernel that serves a call only where default_splits would cut its rows."""
    lib = D.L.lib()
    for q, kv in ((torch.float16, torch.int8), (torch.bfloat16, torch.bfloat16)):
        for n in (0, 1, 2, 64, 127, 128, 129, 255, 256, 257, 5000):
            for ctx in (*range(0, 6000, 61), 511, 512, 767, 768, 999, 1000, 1024, 2900, 100000):
                if lib.uvmi_default_splits(n, ctx, 256) == 1:
                    assert lib.uvmi_decode_attn_splits(D.L.dtype_code(q), D.L.dtype_code(kv), n, 8, 64, 1 << 20, 0, ctx, 256) == 1


def test_splits_of_a_compiled_call(monkeypatch):
    """torch.compile takes the whole call, and cuts it by its strides."""
    monkeypatch.setattr(D, "_device_cus", lambda index: 256)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(D.L, "require_cuda", lambda *t: None)
    taken = []

    def backend(gm, example):
        taken.extend(n.args[10] for n in gm.graph.nodes if "decode_attn" in str(n.target))
        return lambda *a: (torch.zeros(2, 8, 64),)
    q, pos = torch.zeros(2, 8, 64).half(), torch.zeros(2, dtype=torch.long)
    for pitch in (64, 68):
        torch._dynamo.reset()
        torch.compile(lambda k: D.decode_attention(q, k, k, pos, pos, 0.1), backend=backend, fullgraph=True)(_cache(torch.float16, 2048, pitch))
    assert taken == [D._own_splits(torch.float16, torch.float16, 2, 8, 64, 2048, False, 2048), D.default_splits(2, 2048)]


@pytest.mark.parametrize("V,d,n,of", [(32768, 640, 1, 1), (32768, 640, 65536, 1 << 20), (32768, 640, 65537, 65537), (32768, 640, 64, (1 << 29) // 640 - 64),
                                      (32768, 640, 64, (1 << 20) + 1), (524288, 1024, 8, 8), (524224, 1024, 8, 8), (524208, 1024, 8, 8), (4096, 8192, 65536, 65536),
                                      (4096, 8192, 65472, 65472), (4096, 8192, 65471, 65471), (4096, 8256, 8, 8), (4096, 96, 8, 8), (4104, 640, 8, 8), (4096, 64, 8, 8)])
def test_logits_of_raw_hidden_are_asked_for_where_the_library_takes_them(V, d, n, of):
    # (beyond, the logits come from the normed hidden as they did: a vocabulary or hidden past 32-bit offsets is no error)
    from types import SimpleNamespace

    from ultraviolet_amd import _lib as L
    from ultraviolet_amd.engine.model import UVEngine
    from ultraviolet_amd.kernels.gemm import SOFTCAP
    W = torch.empty(V, d, dtype=torch.bfloat16, device="meta")
    e = SimpleNamespace(w=SimpleNamespace(embed=W), dtype=torch.bfloat16)
    e._own_logits_ok = lambda dtype: UVEngine._own_logits_ok(e, dtype)
    lib = lambda rows: L.lib().uvmi_gemm_tn_supported(L.dtype_code(W.dtype), rows, V, d, d, d, V, SOFTCAP) == 1
    takes = lib(n) and d >= 128 and (of == n or (of <= 1 << 20 and (of + 64) * d * 2 < 1 << 30))   # (uvmi_head's line for a gathered hidden)
    assert UVEngine._raw_logits_ok(e, n, of) == takes


@pytest.mark.parametrize("d", [192, 256, 640, 1024, 1088])
@pytest.mark.parametrize("H,f", [(1, 640), (2, 640), (8, 64), (8, 128), (1, 64), (8, 1664), (128, 8192)])
@pytest.mark.parametrize("n", [12287, 12288, 40000, 65536, 65537])
def test_passes_keep_sums_of_squares_where_the_library_takes_all_four_products(d, H, f, n):
    """A width that uvmi_gemm_sums refuses for one of them runs as it did without.  (Asked with sums that lie where they may not, the library answers for the
    shape first and launches nothing.)"""
    from types import SimpleNamespace as N

    from ultraviolet_amd import _lib as L
    from ultraviolet_amd.engine.model import UVEngine
    from ultraviolet_amd.engine.weights import UVWeights
    from ultraviolet_amd.kernels.gemm import RESID, STORE, SWIGLU
    cfg = N(d_model=d, n_heads=H, n_kv_heads=1, head_dim=64, d_ff=f)
    e = N(cfg=cfg, big_rows=12288, fold_qkv_rows=1 << 17, gemm_config=0)
    ext = UVWeights.qkv_ext_rows(cfg)

    def refused(epilogue, cols, K, out, norm):
        g = L.GemmArgs(a=256, w=256, c=256, dtype=L.dtype_code(torch.bfloat16), M=n, N=cols, K=K, lda=K, ldw=K, ldc=out, epilogue=epilogue, norm_a=norm, eps=1e-6,
                       resid=256 if epilogue == RESID else None, ldr=out)
        return L.lib().uvmi_gemm_sums(ctypes.byref(L.GemmSumsArgs(ctypes.addressof(g), 4, 1 << 17)), None) == -2
    takes = not any(refused(*p) for p in [(STORE, ext, d, ext, 1), (RESID, d, H * 64, d, 0), (SWIGLU, 2 * f, d, f, 1), (RESID, d, f, d, 0)])
    assert UVEngine._sums_ok(e, n) == takes or (n == 65536 and f == 8192)   # (which no product of this library takes, with sums or without)


@pytest.mark.parametrize("M,N,K,tile", [(12288, 256, 256, 0), (16000, 256, 640, 0), (24576, 256, 2048, 0), (32768, 256, 512, 0), (33216, 256, 512, 192), (16000, 64, 512, 0),
                                        (40000, 128, 1664, 0), (21760, 384, 1024, 0), (22000, 384, 1024, 192), (13056, 640, 512, 0), (14000, 640, 512, 192), (18432, 640, 1664, 192)])
def test_residual_updates_of_one_round_keep_the_smaller_tiles(M, N, K, tile):
    """192 x 128 tiles are for updates whose 128 x 128 ones are more than a round of the device (512 of them on 256 compute units)."""
    from ultraviolet_amd import _lib as L
    from ultraviolet_amd.kernels.gemm import RESID
    g = L.GemmArgs(a=256, w=256, c=256, dtype=L.dtype_code(torch.bfloat16), M=M, N=N, K=K, lda=K, ldw=K, ldc=N, epilogue=RESID, resid=256, ldr=N)
    assert L.lib().uvmi_gemm_resid_tile(ctypes.byref(g)) == tile


def test_guard_of_recorded_passes_sees_what_changes():
    """Everything that launches took an address or a number from: a tensor replaced, moved under its object, a scalar, an entry that
    comes or goes - in the weights and in the state; by torch's comparison of addresses and by the list of them."""
    from types import SimpleNamespace as N
    from ultraviolet_amd.engine import plan
    t = lambda: torch.zeros(4)
    w = N(embed=t(), value_embed=None, inv_freq=t(), layers=[{"wo": t(), "wqkv": t(), "xsa": None, "resid_attn": 1.5} for _ in range(2)])
    st = N(k=[t(), t()], v=[t(), t()], k_scale=[None, None], v_scale=[None, None])

    def moved(x):
        x.data = x.data.clone()
    changes = [lambda: setattr(w, "embed", t()), lambda: moved(w.embed), lambda: moved(w.inv_freq), lambda: setattr(w, "value_embed", t()),
               lambda: w.layers[1].__setitem__("wo", t()), lambda: moved(w.layers[0]["wo"]), lambda: w.layers[0].__setitem__("resid_attn", w.layers[0]["resid_attn"] + 1.0),
               lambda: w.layers[0].__setitem__("xsa", t()), lambda: w.layers[1].__setitem__("new", t()), lambda: w.layers[1].pop("new"),
               lambda: w.layers[0].__setitem__("wqkv", t()), lambda: st.k.__setitem__(1, t()), lambda: moved(st.v[0]), lambda: st.v.pop()]
    same = plan._same_addresses
    try:
        for f in (same, lambda ts, at, _: list(map(torch.Tensor.data_ptr, ts)) == at):
            plan._same_addresses = f
            for change in changes if f is same else changes[:9]:
                g = plan.Guard(w, st)
                assert g.holds(w, st)
                change()
                assert not g.holds(w, st)
            if f is same:
                st.v.append(t())
                w.value_embed = None
    finally:
        plan._same_addresses = same


def test_native_path_sees_what_plain_eager_sees():
    """csrc/eager.cpp asks plain_eager's questions itself, but for the two that decode_attention asks before it."""
    native = D.L.eager().plain
    q, k, v = _qkv()
    ks = vs = torch.ones(2, 1, 32).half()
    calls = [(q, k, v, None, None), (q, k, v, ks, vs), (q, k, v, None, vs), (q.clone().requires_grad_(), k, v, ks, vs), (q, k, v, ks.clone().requires_grad_(), vs),
             (q, k.as_subclass(_Subclass), v, ks, vs), (q, k, v, ks, vs.as_subclass(_Subclass)), (q, torch.nn.Parameter(k), v, None, None),
             (q, torch.nn.Parameter(k, requires_grad=False), v, None, None)]

    def same():
        return [native(*c) for c in calls] == [D.plain_eager(*c) for c in calls]
    assert native(*calls[0]) and native(*calls[1]) and not any(native(*c) for c in calls[3:])
    assert same()
    with torch.inference_mode():
        assert native(*calls[1]) and same()
    with torch.no_grad():
        assert native(*calls[1]) and same()
    with _Passing():
        assert not native(*calls[1]) and same()
    with torch.overrides.BaseTorchFunctionMode():
        assert not native(*calls[1]) and same()
    seen = []
    torch.func.vmap(lambda a: (seen.append((native(a, k, v, ks, vs), D.plain_eager(a, k, v, ks, vs))), a)[1])(q[None])
    torch.func.grad(lambda a: (seen.append((native(a, k, v, ks, vs), D.plain_eager(a, k, v, ks, vs))), a.sum())[1])(q.float())
    assert seen == [(False, False)] * 2


def test_native_path_leaves_other_calls_to_the_general_one():
    """None for what is not on a device, and nothing raised: the general path has its own words for it."""
    q, k, v = _qkv()
    idx = torch.zeros(2, dtype=torch.long)
    assert D.L.eager().decode_attention(q, k, v, None, None, idx, idx, None, 0.1, 0, None, None, 1, False, 0) is None
    assert D.L.eager().decode_attention(q, k, 3, None, None, idx, None, None, 0.1, 0, None, None, 1, False, 0) is None


def test_native_path_of_another_build_is_not_loaded(monkeypatch, tmp_path):
    """The extension is looked for under the interpreter's and torch's versions, refused when it was built for another revision of the
    argument structs or calls a library of one, and where there is none the general path takes every call."""
    import sysconfig
    L = D.L
    q, k, v = _qkv()
    idx = torch.zeros(2, dtype=torch.long)
    assert sysconfig.get_config_var("SOABI") in L.EAGER_PATH and torch.__version__ in L.EAGER_PATH
    mod = L.eager()
    assert mod.revision == mod.library_revision == L.ABI_VERSION and mod.attn_args_bytes == ctypes.sizeof(L.AttnArgs)

    def none_of_it(words):
        monkeypatch.setattr(L, "_eager", None)
        with pytest.raises(L.UvmiError, match=words):
            L.eager()
        D._native.cache_clear()
        with pytest.warns(UserWarning, match=words):
            native = D._native()
        D._native.cache_clear()
        assert native(q, k, v, None, None, idx, idx, None, 0.1, 0, None, None, 1, False, 0) is None
    with monkeypatch.context() as m:
        m.setattr(L, "ABI_VERSION", L.ABI_VERSION + 1)
        none_of_it("revision")
    with monkeypatch.context() as m:
        m.setattr(L, "AttnArgs", L.SampleArgs)
        none_of_it("revision")
    with monkeypatch.context() as m:
        m.setattr(L, "EAGER_PATH", str(tmp_path / "none.so"))
        none_of_it("not found")
    with monkeypatch.context() as m:
        (tmp_path / "other.so").write_bytes(b"not a library")
        m.setattr(L, "EAGER_PATH", str(tmp_path / "other.so"))
        none_of_it("does not load")


@pytest.mark.parametrize("lacks", ["prefill_attn_args_bytes", "varlen_attention", "revision"])
def test_native_path_that_lacks_something_is_another_build(monkeypatch, lacks):
    """An extension without what this one asks it for is refused as one of another revision is, and calls take the general path."""
    from types import SimpleNamespace as N

    from ultraviolet_amd.kernels import varlen_attn as V
    L = D.L
    real = L.eager()
    old = N(**{a: getattr(real, a) for a in dir(real) if not a.startswith("__") and a != lacks})
    monkeypatch.setattr(L, "_eager", None)
    monkeypatch.setattr(L.importlib.util, "spec_from_file_location", lambda *a: N(loader=N(exec_module=lambda m: None)))
    monkeypatch.setattr(L.importlib.util, "module_from_spec", lambda spec: old)
    with pytest.raises(L.UvmiError, match="rebuild"):
        L.eager()
    for native, n in ((D._native, 15), (V._native, 6)):
        native.cache_clear()
        with pytest.warns(UserWarning, match="rebuild"):
            assert native()(*[None] * n) is None
        native.cache_clear()


def test_library_that_lacks_an_entry_point_is_refused(monkeypatch):
    from types import SimpleNamespace as N
    L = D.L
    monkeypatch.setattr(L, "_lib", None)
    monkeypatch.setattr(L.C, "CDLL", lambda path: N(uvmi_version=lambda: L.ABI_VERSION))
    with pytest.raises(L.UvmiError, match="uvmi_decode_attn_splits.*rebuild"):
        L.lib()


def test_library_is_built_where_the_extension_cannot_be(monkeypatch, tmp_path, capsys):
    """A compiler or headers that are missing cost the extension only, and an older one does not stay."""
    from ultraviolet_amd.csrc import build as B
    old = tmp_path / "eager.so"
    old.write_bytes(b"older")
    monkeypatch.setattr(D.L, "EAGER_PATH", str(old))

    def run(cmd):
        raise RuntimeError("no such header")
    B._build_eager(run, True, True)
    assert not old.exists() and "no such header" in capsys.readouterr().err
    monkeypatch.setenv("CXX", str(tmp_path / "no-compiler"))
    B._build_eager(lambda cmd: subprocess.run(cmd, check=True), True, True)
    assert "no-compiler" in capsys.readouterr().err
