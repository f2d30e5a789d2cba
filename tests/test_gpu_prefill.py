"""GPU parity: packed causal / windowed prefill attention (uvmi_prefill_attn through the C ABI) vs the CPU oracle.

The first case restates the reference's own test (tests/test_perf_opt.py:40-61, forward part): segment lengths
[300, 1000, 57, 700, 1], 8 query heads on 1 kv head, head_dim 64, fp16, window None / 256, |o - ref|.max() < 2e-3.
With fp16 inputs the probabilities are rounded to fp16 before P.V (as in the reference's tensor-core kernel); with bf16
inputs they are rounded to bf16, which bounds the error by 2^-9 * sum p|v| instead, so that case carries a 4e-3 bar."""
import numpy as np
import pytest
import torch

from util import to_np

pytestmark = pytest.mark.gpu
DEV = "cuda"
SC = 1.13 / 8


def _case(lens, H, K, hd, dtype, seed=0, kv_dtype=None):
    g = torch.Generator().manual_seed(seed)
    N = int(sum(lens))
    q = torch.randn(N, H, hd, generator=g).to(dtype)
    k = torch.randn(N, K, hd, generator=g).to(kv_dtype or dtype)
    v = torch.randn(N, K, hd, generator=g).to(kv_dtype or dtype)
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    return q, k, v, cu


def _check(q, k, v, cu, window, atol, expect_path=None, scale=SC):
    from oracle.varlen_attn import varlen_attention_ref
    from ultraviolet_amd.kernels.varlen_attn import packed_attention, packed_attention_path
    d = lambda t: t.to(DEV)
    qd, kd, vd, cud = d(q), d(k), d(v), d(cu)
    if expect_path is not None:
        assert packed_attention_path(qd, kd, vd, cud, scale, window) == expect_path
    o32 = packed_attention(qd, kd, vd, cud, scale, window, out_fp32=True)
    o = packed_attention(qd, kd, vd, cud, scale, window)
    torch.cuda.synchronize()
    ref = varlen_attention_ref(to_np(q), to_np(k), to_np(v), to_np(cu), scale, window)
    a32, a = to_np(o32), to_np(o)
    assert np.isfinite(a32).all()
    assert np.abs(a32 - ref).max() < atol, np.abs(a32 - ref).max()
    out_eps = 2.0 ** -11 if q.dtype == torch.float16 else 2.0 ** -8
    assert np.abs(a - ref).max() < atol + out_eps * np.abs(ref).max()
    return a32, ref


@pytest.mark.parametrize("window", [None, 256])
def test_reference_case_fp16(window):
    q, k, v, cu = _case([300, 1000, 57, 700, 1], 8, 1, 64, torch.float16)
    from ultraviolet_amd.kernels import varlen_attention
    a32, ref = _check(q, k, v, cu, window, 2e-3, expect_path=1)
    o = varlen_attention(q[None].to(DEV), k[None].to(DEV), v[None].to(DEV), cu.to(DEV), 1000, SC, window)
    assert o.shape == (1, q.size(0), 8, 64) and o.dtype == torch.float16
    assert (o[0].float().cpu().numpy() - ref).__abs__().max() < 2e-3   # the reference's bar on the fp16 output


@pytest.mark.parametrize("window", [None, 256])
def test_reference_case_bf16(window):
    q, k, v, cu = _case([300, 1000, 57, 700, 1], 8, 1, 64, torch.bfloat16, seed=1)
    _check(q, k, v, cu, window, 4e-3, expect_path=1)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens", [[1], [15], [16], [17], [1, 1, 1, 1, 1], [0, 5, 0, 0, 40, 0], [31, 33, 64, 1, 2, 95, 7],
                                  [512] * 3, [3, 700, 2]])
@pytest.mark.parametrize("window", [None, 1, 16, 33, 256])
def test_ragged_and_edges(dtype, lens, window):
    q, k, v, cu = _case(lens, 8, 1, 64, dtype, seed=len(lens))
    _check(q, k, v, cu, window, 2e-3 if dtype == torch.float16 else 4e-3, expect_path=1)


@pytest.mark.parametrize("tiles", range(1, 10))
@pytest.mark.parametrize("H,window", [(8, None), (5, 40), (4, None), (2, 40)])
def test_even_and_odd_counts_of_key_tiles(tiles, H, window):
    # (one sequence's last block walks every count of 32-key tiles, the sequence behind it starts inside a tile; bars as above)
    q, k, v, cu = _case([32 * tiles - 3, 32 * tiles + 1], H, 1, 64, torch.float16, seed=tiles)
    _check(q, k, v, cu, window, 2e-3, expect_path=1)


@pytest.mark.parametrize("n_seg", [1, 2, 63, 64, 65])
@pytest.mark.parametrize("H,first,idx", [(8, 0, torch.int32), (4, 3, torch.int64), (2, 40, torch.int32)])
def test_segment_table_of_few_and_many_sequences(n_seg, H, first, idx):
    """Up to 64 sequences, empty ones among them, the attention finds its rows' sequences itself; the table that it leaves is the one of the launch for more
    of them, which the same boundaries with empty sequences behind them get."""
    from ultraviolet_amd.kernels.varlen_attn import packed_attention
    r = np.random.default_rng(n_seg)
    lens = r.integers(0, 20, size=n_seg) + (n_seg == 1)
    N = first + int(lens.sum()) + 5   # (tokens ahead of the first sequence and behind the last)
    cu = torch.from_numpy(first + np.concatenate([[0], np.cumsum(lens)])).to(idx)
    many = torch.cat([cu, cu[-1:].expand(70)])
    q, k, v, _ = (t.to(DEV) for t in _case([N], H, 1, 64, torch.float16, seed=n_seg))
    got = []
    for c in (cu, many):
        ws = torch.zeros(2 * ((4 * N + 255) // 256 * 256), dtype=torch.uint8, device=DEV)
        got.append((packed_attention(q, k, v, c.to(DEV), SC, 30, workspace=ws), ws))
    seg = [w.view(torch.int32)[:N].cpu().numpy() for _, w in got]
    c, i = cu.numpy(), np.arange(N)
    want = c[np.maximum(np.searchsorted(c[:-1], i, side="right") - 1, 0)]
    assert (seg[0] == np.where(want <= i, want, i + 1)).all()
    end = int(cu[-1])   # (what follows the last sequence belongs to the empty ones in `many`)
    assert (seg[0][:end] == seg[1][:end]).all() and torch.equal(got[0][0][:end], got[1][0][:end])


@pytest.mark.parametrize("H", [8, 4, 2])
def test_tiles_outside_a_blocks_keys_are_not_touched(H):
    # (NaN in the values of a sequence whose tiles no other sequence's rows share stays in that sequence)
    q, k, v, cu = _case([64, 32, 96, 32, 32], H, 1, 64, torch.float16)
    from ultraviolet_amd.kernels.varlen_attn import packed_attention
    clean = packed_attention(*(t.to(DEV) for t in (q, k, v, cu)), SC)
    v[64:96] = float("nan")
    v[192:224] = float("nan")
    got = packed_attention(*(t.to(DEV) for t in (q, k, v, cu)), SC)
    for a, b in ((0, 64), (96, 192), (224, 256)):
        assert torch.equal(got[a:b], clean[a:b])
    assert got[64:96].isnan().all() and got[192:224].isnan().all()


@pytest.mark.parametrize("H,K", [(1, 1), (4, 1), (5, 1), (8, 2), (6, 2), (16, 2), (8, 8)])
def test_head_groupings(H, K):
    q, k, v, cu = _case([40, 130, 9], H, K, 64, torch.float16, seed=H * 10 + K)
    _check(q, k, v, cu, 64, 2e-3, expect_path=1)


def test_strided_views_of_one_buffer_and_int64_cu():
    """q, k, v as column slices of one (N, (H + 2K) * hd) projection output, as a fused QKV GEMM leaves them."""
    from oracle.varlen_attn import varlen_attention_ref
    from ultraviolet_amd.kernels.varlen_attn import packed_attention, packed_attention_path
    H, K, hd, lens = 8, 1, 64, [100, 37, 260]
    N = sum(lens)
    g = torch.Generator().manual_seed(5)
    qkv = torch.randn(N, (H + 2 * K) * hd, generator=g).to(torch.bfloat16).to(DEV)
    q = qkv[:, :H * hd].view(N, H, hd)
    k = qkv[:, H * hd:(H + K) * hd].view(N, K, hd)
    v = qkv[:, (H + K) * hd:].view(N, K, hd)
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int64, device=DEV)
    assert packed_attention_path(q, k, v, cu, SC, 256) == 1
    o = packed_attention(q, k, v, cu, SC, 256, out_fp32=True)
    ref = varlen_attention_ref(to_np(q), to_np(k), to_np(v), to_np(cu), SC, 256)
    assert np.abs(to_np(o) - ref).max() < 4e-3


@pytest.mark.parametrize("hd,kv_dtype", [(64, torch.float32), (128, torch.float16), (32, torch.bfloat16)])
def test_generic_path(hd, kv_dtype):
    """fp32 K/V (an fp32 engine keeps q in fp16) and other head dims run the VALU kernel, token by token."""
    qd = torch.float16 if kv_dtype != torch.bfloat16 else torch.bfloat16
    q, k, v, cu = _case([33, 1, 90], 4, 1, hd, qd, seed=3, kv_dtype=kv_dtype)
    _check(q, k, v, cu, 48, 2e-3, expect_path=0, scale=1.0 / np.sqrt(hd))


def test_exact_special_cases():
    """V == 1 gives exactly 1 wherever a row sees any key (sum p~ / sum p, both from the same rounded values up to 2^-11);
    window 1 returns the row's own v (softmax over one key is 1)."""
    from ultraviolet_amd.kernels.varlen_attn import packed_attention
    q, k, v, cu = _case([200, 56, 300], 8, 1, 64, torch.float16, seed=9)
    d = lambda t: t.to(DEV)
    ones = torch.ones_like(v)
    o = packed_attention(d(q), d(k), d(ones), d(cu), SC, 128, out_fp32=True)
    assert np.abs(to_np(o) - 1.0).max() < 1e-3
    o = packed_attention(d(q), d(k), d(v), d(cu), SC, 1, out_fp32=True)
    # p = exp2(fma(s, c, -round(s c))) is 1 up to an ulp, so the normaliser is too
    np.testing.assert_allclose(to_np(o), np.broadcast_to(to_np(v).astype(np.float32), o.shape), rtol=1e-6, atol=0)


@pytest.mark.parametrize("window", [0, 256])
def test_mixed_batch_chunk_shape(window):
    """The prefill half of the mixed-batch configuration: 64 chunks x 512 tokens, bf16, 8 heads on 1 kv head.  The oracle
    checks 3 of the chunks; all chunks see statistically identical inputs, and identical inputs give identical outputs:
    chunk 5 is a copy of chunk 4 shifted by one 512-token (block-aligned) segment, so its output must be bit-identical."""
    from oracle.varlen_attn import varlen_attention_ref
    from ultraviolet_amd.kernels.varlen_attn import packed_attention
    lens = [512] * 64
    q, k, v, cu = _case(lens, 8, 1, 64, torch.bfloat16, seed=11)
    for t in (q, k, v):
        t[5 * 512:6 * 512] = t[4 * 512:5 * 512]
    o = to_np(packed_attention(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), SC, window, out_fp32=True))
    assert np.isfinite(o).all()
    np.testing.assert_array_equal(o[5 * 512:6 * 512], o[4 * 512:5 * 512])
    for s in (0, 4, 63):
        sl = slice(s * 512, (s + 1) * 512)
        ref = varlen_attention_ref(to_np(q[sl]), to_np(k[sl]), to_np(v[sl]), [0, 512], SC, window)
        assert np.abs(o[sl] - ref).max() < 4e-3


def test_error_paths():
    from ultraviolet_amd import _lib as L
    from ultraviolet_amd.kernels.varlen_attn import packed_attention
    q, k, v, cu = _case([20], 8, 1, 64, torch.float16)
    with pytest.raises(L.UvmiError):
        packed_attention(q, k, v, cu, SC)                       # host tensors
    d = lambda t: t.to(DEV)
    with pytest.raises((L.UvmiError, KeyError)):
        packed_attention(d(q).double(), d(k), d(v), d(cu), SC)   # queries are fp16, bf16 or fp32
    o32 = packed_attention(d(q).float(), d(k).float(), d(v).float(), d(cu), SC)   # fp32 throughout: the plain fp32 kernel
    o16 = packed_attention(d(q), d(k), d(v), d(cu), SC, out_fp32=True)
    assert o32.dtype == torch.float32 and (o32 - o16).abs().max() < 2e-3
    with pytest.raises(AssertionError):
        packed_attention(d(q), d(k), d(v), d(cu), SC, workspace=torch.empty(64, dtype=torch.uint8, device=DEV))  # too small


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("window", [0, 48])
def test_packed_attention_fused_post_epilogue(dtype, window):
    """post=(vhat, gate, xsa): the kernel's epilogue equals Attention.post applied to its own plain output
    (ultraviolet/model.py:321-333: z -= xsa_h (z . v_hat) v_hat on the output rounded to the activation type, then the
    per-head gate), evaluated here in float64 from the plain output of the same kernel; reusing the segment table of an
    earlier call (segments_ready) changes nothing."""
    from ultraviolet_amd.kernels.varlen_attn import packed_attention
    g = torch.Generator(device="cuda").manual_seed(5)
    lens = [37, 1, 160, 64, 5]
    N, H, K, hd = sum(lens), 8, 2, 64
    cu = torch.tensor([0] + list(np.cumsum(lens)), device="cuda")
    q = torch.randn(N, H, hd, device="cuda", generator=g).to(dtype)
    k = torch.randn(N, K, hd, device="cuda", generator=g).to(dtype)
    v = torch.randn(N, K, hd, device="cuda", generator=g).to(dtype)
    vhat = torch.nn.functional.normalize(v.float(), dim=-1).contiguous()
    gate = (torch.rand(N, H, device="cuda", generator=g) * 2).contiguous()
    xsa = torch.tanh(torch.randn(H, device="cuda", generator=g)).contiguous()
    ws = torch.empty(1 << 16, dtype=torch.uint8, device="cuda")
    plain = packed_attention(q, k, v, cu, 0.125, window, workspace=ws)
    fused = packed_attention(q, k, v, cu, 0.125, window, workspace=ws, segments_ready=True, post=(vhat, gate, xsa))
    z = plain.double()
    vh = vhat.double().repeat_interleave(H // K, dim=1)
    want = (z - xsa.double()[None, :, None] * (z * vh).sum(-1, keepdim=True) * vh) * gate.double()[:, :, None]
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    err = (fused.double() - want).abs()
    assert float((err / (want.abs() + 1.0)).max()) <= 3 * ulp, float((err / (want.abs() + 1.0)).max())
    no_gate = packed_attention(q, k, v, cu, 0.125, window, workspace=ws, post=(vhat, None, None))
    assert float((no_gate.double() - z).abs().max()) <= 2 * ulp * float(z.abs().max())


def _grad_case(lens, H, K, dtype, window, seed=0):
    from oracle.varlen_attn import varlen_attention_grad_ref
    from ultraviolet_amd.kernels import varlen_attention
    q, k, v, cu = _case(lens, H, K, 64, dtype, seed=seed)
    go = torch.randn(q.shape, generator=torch.Generator().manual_seed(seed + 100)).to(dtype)
    qd, kd, vd = (t[None].to(DEV).requires_grad_() for t in (q, k, v))
    o = varlen_attention(qd, kd, vd, cu.to(DEV), max(max(lens), 1), SC, window)
    o.backward(go[None].to(DEV))
    torch.cuda.synchronize()
    ref = varlen_attention_grad_ref(to_np(q), to_np(k), to_np(v), to_np(go), to_np(cu), SC, window)
    got = [to_np(t.grad[0]).astype(np.float64) for t in (qd, kd, vd)]
    return got, ref


@pytest.mark.parametrize("window", [None, 256])
def test_backward_reference_case_fp16(window):
    """The reference's own test of the varlen backward (tests/test_perf_opt.py:40-61): lens [300, 1000, 57, 700, 1], 8 query
    heads on 1 kv head, fp16, window None / 256, gradients through autograd; its bar: |g - g_ref| / |g_ref| < 5e-3 for each
    of dq, dk, dv (norms over the whole tensor)."""
    got, ref = _grad_case([300, 1000, 57, 700, 1], 8, 1, torch.float16, window)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert np.linalg.norm(a - b) / np.linalg.norm(b) < 5e-3, np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens,H,K,window", [([1], 8, 1, None), ([0, 5, 0, 0, 40, 0], 8, 1, 16), ([31, 33, 64, 1, 2, 95, 7], 8, 2, 33),
                                             ([70, 3], 4, 4, 1), ([130], 2, 1, None), ([65, 64, 63], 8, 8, 64)])
def test_backward_ragged_and_edges(dtype, lens, H, K, window):
    """Empty and single-token segments, segment boundaries inside a wave's 64 queries / 32 keys, window 1 (every query sees
    only itself: dq = dk = 0 up to rounding, dv = go summed over the group), grouped and per-head K / V."""
    got, ref = _grad_case(lens, H, K, dtype, window, seed=3)
    ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert np.abs(a - b).max() <= 2 * ulp * max(np.abs(b).max(), 1e-3) + 1e-6, (np.abs(a - b).max(), np.abs(b).max())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,K,window", [(8, 1, None), (8, 2, 256), (4, 1, 100), (16, 1, 64)])
def test_backward_many_tiles_and_padding_tokens(dtype, H, K, window):
    """Sequences of several 32-key tiles and 64-key workgroups (interior tiles take the unmasked path), a group of 16 heads
    (beyond the matrix-core kernels' 8: the plain kernels), and 37 tokens past cu[-1]: padding, whose gradients are zero and
    which no real key may see."""
    from oracle.varlen_attn import varlen_attention_grad_ref
    from ultraviolet_amd.kernels.varlen_attn import packed_attention, packed_attention_backward
    lens, pad = [512, 700, 300, 5], 37
    q, k, v, cu = _case(lens, H, K, 64, dtype, seed=11)
    N = q.size(0)
    gen = torch.Generator().manual_seed(12)
    go = torch.randn(q.shape, generator=gen).to(dtype)
    ext = lambda t: torch.cat([t, torch.randn(pad, *t.shape[1:], generator=gen).to(dtype)]).to(DEV)
    qd, kd, vd, god = ext(q), ext(k), ext(v), ext(go)
    o = packed_attention(qd, kd, vd, cu.to(DEV), SC, window)
    dq, dk, dv = packed_attention_backward(god, qd, kd, vd, o, cu.to(DEV), SC, window)
    torch.cuda.synchronize()
    ref = varlen_attention_grad_ref(to_np(q), to_np(k), to_np(v), to_np(go), to_np(cu), SC, window)
    ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    for a, b in zip((dq, dk, dv), ref):
        a = to_np(a).astype(np.float64)
        assert np.isfinite(a).all() and (a[N:] == 0).all()
        assert np.abs(a[:N] - b).max() <= 2 * ulp * np.abs(b).max() + 1e-6, (np.abs(a[:N] - b).max(), np.abs(b).max())
        assert np.linalg.norm(a[:N] - b) / np.linalg.norm(b) < (5e-3 if dtype == torch.float16 else 2e-2)


@pytest.mark.parametrize("H,K", [(3, 1), (7, 1), (10, 2)])
@pytest.mark.parametrize("n", [32, 33, 63, 65, 97])
def test_backward_odd_head_groups_at_block_edges(H, K, n):
    """Head groups that end inside a pair of heads, with keys and queries that end at and around the edges of the 32- and 64-row
    blocks; a sequence boundary and a window inside a block."""
    for lens, window in (([n], None), ([n - 20, 20], 24)):
        got, ref = _grad_case(lens, H, K, torch.bfloat16, window, seed=n)
        for a, b in zip(got, ref):
            assert np.isfinite(a).all()
            assert np.abs(a - b).max() <= 2 * 2.0 ** -7 * np.abs(b).max() + 1e-6, (lens, np.abs(a - b).max(), np.abs(b).max())


@pytest.mark.parametrize("tiles", range(1, 8))
@pytest.mark.parametrize("H,K,window", [(8, 1, None), (5, 1, 40), (4, 1, None), (6, 2, 40)])
def test_backward_even_and_odd_counts_of_key_tiles(tiles, H, K, window):
    """dq with one and two heads of a wave over every count of 32-key tiles; two roundings of the largest gradient."""
    got, ref = _grad_case([32 * tiles - 3, 32 * tiles + 1], H, K, torch.float16, window, seed=tiles)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert np.abs(a - b).max() <= 2 * 2.0 ** -10 * np.abs(b).max() + 1e-6, (np.abs(a - b).max(), np.abs(b).max())


@pytest.mark.parametrize("window", [2, 31, 32, 33, 64, 65, 96, 97, 330, 331, 332, 2 ** 31 - 1])
def test_attention_and_backward_at_the_mask_rules(window):
    """Windows around the places where a 32-key tile stops needing a mask, or a wave of 32 keys stops seeing a 32-query tile: both
    depend on the window modulo the tile and on the sequence's start and end inside one; and windows that hide one key and none.
    Tolerance: one rounding of the largest value for the forward, two for the gradients (as above)."""
    from oracle.varlen_attn import varlen_attention_ref
    from ultraviolet_amd.kernels import varlen_attention
    lens, ulp = [331, 37, 130], 2.0 ** -10
    q, k, v, cu = _case(lens, 8, 1, 64, torch.float16, seed=5)
    o = varlen_attention(q[None].to(DEV), k[None].to(DEV), v[None].to(DEV), cu.to(DEV), max(lens), SC, window)
    ref = varlen_attention_ref(to_np(q), to_np(k), to_np(v), to_np(cu), SC, window)
    assert np.abs(to_np(o[0]).astype(np.float64) - ref).max() <= ulp * np.abs(ref).max()
    got, ref = _grad_case(lens, 8, 1, torch.float16, window, seed=5)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert np.abs(a - b).max() <= 2 * ulp * np.abs(b).max() + 1e-6, (np.abs(a - b).max(), np.abs(b).max())


@pytest.mark.parametrize("G", [1, 2, 3, 8])
@pytest.mark.parametrize("K,lens,window", [(40, [330, 5, 200], None), (20, [330, 5, 200], 70), (20, [330, 5, 200], None), (1, [3] * 64 + [40], None), (2, [2, 0, 5] * 50, 4)])
def test_backward_of_keys_by_heads_and_strides(G, K, lens, window):
    """dk / dv with more workgroups than the 8-wave form takes (with and without a window) and fewer, for every padding of the head group; around and
    beyond the 64 sequences whose ends a wave holds.  Tolerance as above."""
    got, ref = _grad_case(lens, G * K, K, torch.float16, window, seed=7)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert np.abs(a - b).max() <= 2 * 2.0 ** -10 * np.abs(b).max() + 1e-6, (np.abs(a - b).max(), np.abs(b).max())


@pytest.mark.parametrize("G,K,lens,window", [(8, 1, [64], None), (8, 1, [63], None), (8, 2, [70] * 66, None), (5, 1, [200, 1, 90], 65), (3, 1, [330, 5, 200], 170), (4, 1, [160], None),
                                             (2, 1, [641, 640], None), (2, 1, [900], 700), (1, 1, [1290], None), (1, 2, [1400], 1300), (8, 10, [820, 3], None), (2, 10, [900], None),
                                             (1, 10, [1300], None)])
def test_backward_of_keys_by_mean_sequence_and_window(G, K, lens, window):
    """dk / dv on either side of the lines that give it eight waves a workgroup or four: the mean sequence, cut to the window, for every padding of the head
    group, up to a workgroup per compute unit and beyond.  Tolerance as above."""
    got, ref = _grad_case(lens, G * K, K, torch.float16, window, seed=9)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert np.abs(a - b).max() <= 2 * 2.0 ** -10 * np.abs(b).max() + 1e-6, (np.abs(a - b).max(), np.abs(b).max())


@pytest.mark.parametrize("window", [33, 167, 168, 2 ** 31 - 1])
def test_plain_backward_with_windows_that_hide_few_keys_and_none(window):
    """16 query heads on a kv head, which the plain kernels serve: windows up to the largest that an int holds.  Tolerance as above."""
    got, ref = _grad_case([131, 37], 16, 1, torch.float16, window, seed=6)
    for a, b in zip(got, ref):
        assert np.isfinite(a).all()
        assert np.abs(a - b).max() <= 2 * 2.0 ** -10 * np.abs(b).max() + 1e-6, (np.abs(a - b).max(), np.abs(b).max())


@pytest.mark.parametrize("H,window", [(8, None), (8, 20), (3, None), (16, None), (16, 20)])
@pytest.mark.parametrize("first,lens", [(5, [35, 10]), (15, [1, 70]), (33, [100]), (130, [40, 64])])
def test_tokens_ahead_of_the_first_sequence_see_nothing(first, lens, H, window):
    """cu_seqlens that begin behind token 0: the tokens ahead of it give zeros, as the definition has them, in the output and in the gradients, whether
    their block of 16 holds tokens of the first sequence or not; the others are untouched by them.  Tolerances as above."""
    from oracle.varlen_attn import varlen_attention_grad_ref, varlen_attention_ref
    from ultraviolet_amd.kernels.varlen_attn import packed_attention, packed_attention_backward
    q, k, v, cu = _case([first] + lens, H, 1, 64, torch.float16, seed=9)
    cu, go, ulp = cu[1:].contiguous(), torch.randn(q.shape, generator=torch.Generator().manual_seed(10)).half(), 2.0 ** -10
    qd, kd, vd, cd, gd = (t.to(DEV) for t in (q, k, v, cu, go))
    o = packed_attention(qd, kd, vd, cd, SC, window)
    ref = varlen_attention_ref(to_np(q), to_np(k), to_np(v), to_np(cu), SC, window)
    assert bool((o[:first] == 0).all()) and np.abs(to_np(o).astype(np.float64) - ref).max() <= ulp * np.abs(ref).max()
    refs = varlen_attention_grad_ref(to_np(q), to_np(k), to_np(v), to_np(go), to_np(cu), SC, window)
    for grad, ref in zip(packed_attention_backward(gd, qd, kd, vd, o, cd, SC, window), refs):
        assert bool((grad[:first] == 0).all()) and np.abs(to_np(grad).astype(np.float64) - ref).max() <= 2 * ulp * np.abs(ref).max() + 1e-6


def test_backward_from_statistics_of_a_wide_pitch():
    """The forward's statistics as rows of a larger array, 8 of them within 32-bit byte offsets and beyond: the bits of the call whose rows are
    close together."""
    from ultraviolet_amd.kernels.varlen_attn import packed_attention, packed_attention_backward, statistics_pitch
    from ultraviolet_amd import _lib as L
    q, k, v, cu = (t.to(DEV) for t in _case([131, 37], 8, 1, 64, torch.bfloat16, seed=7))
    go = torch.randn(q.shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(8)).to(q.dtype)
    N, grads = q.size(0), []
    ws = torch.empty(L.lib().uvmi_prefill_attn_workspace_bytes(N), dtype=torch.uint8, device=DEV)
    for pitch in (statistics_pitch(N), 1 << 20, 160_000_000):
        lse = torch.empty(7 * pitch + statistics_pitch(N), device=DEV).as_strided((8, statistics_pitch(N)), (pitch, 1))
        o = packed_attention(q, k, v, cu, SC, 100, workspace=ws, lse_out=lse)
        grads.append(packed_attention_backward(go, q, k, v, o, cu, SC, 100, saved=(lse, ws)))
    for other in grads[1:]:
        assert all(torch.equal(a, b) for a, b in zip(grads[0], other))


def test_backward_rejects_what_it_cannot_do():
    from ultraviolet_amd import _lib as L
    from ultraviolet_amd.kernels.varlen_attn import packed_attention_backward
    cu = torch.tensor([0, 4], dtype=torch.int32, device=DEV)
    z = lambda *s_, dt=torch.float16: torch.zeros(*s_, dtype=dt, device=DEV)
    with pytest.raises(L.UvmiError):   # head_dim 32
        packed_attention_backward(z(4, 2, 32), z(4, 2, 32), z(4, 1, 32), z(4, 1, 32), z(4, 2, 32), cu, 1.0)
    with pytest.raises(L.UvmiError):   # fp32 tensors
        packed_attention_backward(*(z(4, 2, 64, dt=torch.float32) for _ in range(2)), *(z(4, 1, 64, dt=torch.float32) for _ in range(2)),
                                  z(4, 2, 64, dt=torch.float32), cu, 1.0)


@pytest.mark.parametrize("form", ["plain", "fp16", "indices64", "views", "padding", "k alone", "no gradient", "no grad mode", "inference", "hooks",
                                  "parameter", "generic", "scale int", "fp32"])
def test_native_varlen_call_equals_the_general_one(monkeypatch, form):
    """varlen_attention's native path (csrc/eager.cpp) and the general one make the same launches on the same arguments: equal bits, output and
    gradients, over the forms a call may take; the last four the native path hands on.  A hook on saved tensors sees the same ones."""
    from ultraviolet_amd.kernels import varlen_attn as A
    dtype = torch.float16 if form == "fp16" else torch.float32 if form == "fp32" else torch.bfloat16
    q, k, v, cu = (t.to(DEV) for t in _case([131, 0, 37, 64], 16 if form == "generic" else 8, 1, 64, dtype, seed=3))
    q, k, v = (t[None] for t in (q, k, v))
    go = torch.randn(q.shape, device=DEV, generator=torch.Generator(device=DEV).manual_seed(4)).to(dtype)
    scale = 1 if form == "scale int" else 0.14
    if form == "indices64":
        cu = cu.long()
    elif form == "views":
        qkv = torch.cat([q, k, v], 2)
        q, k, v, go = qkv[:, :, :8], qkv[:, :, 8:9], qkv[:, :, 9:], go.transpose(1, 2).contiguous().transpose(1, 2)
    elif form == "padding":
        cu = cu[:3].contiguous()
    elif form == "parameter":
        q = torch.nn.Parameter(q)
    grads = form not in ("no gradient", "no grad mode", "inference", "generic", "fp32")
    wrt = [k] if form == "k alone" else [q, k, v]
    if form != "no gradient" and form != "generic" and form != "fp32":
        wrt = [t.detach().requires_grad_() if form != "parameter" or t is not q else t for t in wrt]
        q, k, v = (q, wrt[0], v) if form == "k alone" else wrt
    seen = []

    def call():
        seen.append([])
        keep = lambda t: seen[-1].append((t.shape, t.dtype)) or t
        with torch.autograd.graph.saved_tensors_hooks(keep, lambda t: t) if form == "hooks" else torch.inference_mode(form == "inference"):
            with torch.set_grad_enabled(form != "no grad mode" and form != "inference"):
                o = A.varlen_attention(q, k, v, cu, 131, scale, 100)
        return (o.detach(), *torch.autograd.grad(o, wrt, go)) if grads else (o,)
    used = []
    native = A._native()
    monkeypatch.setattr(A, "_native", lambda: lambda *a: used.append(native(*a)) or used[-1])
    got = call()
    monkeypatch.setattr(A, "_native", lambda: lambda *a: None)
    want = call()
    assert (used[0] is None) == (form in ("parameter", "generic", "scale int", "fp32"))
    assert len(got) == len(want) and all(a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b) for a, b in zip(got, want))
    assert seen[0] == seen[1] and (form != "hooks" or len(seen[0]) == 7)


def test_native_varlen_gradient_of_a_changed_input_is_refused():
    """A saved operand changed in place before the backward: the error of a graph, not gradients of other values."""
    from ultraviolet_amd.kernels import varlen_attention
    q, k, v, cu = (t.to(DEV) for t in _case([64, 7], 8, 1, 64, torch.bfloat16, seed=3))
    q, k, v = (t[None] for t in (q, k, v))
    q.requires_grad_()
    o = varlen_attention(q, k, v, cu, 64, 0.14)
    k.add_(1)
    with pytest.raises(RuntimeError, match="inplace"):
        o.sum().backward()
    o = varlen_attention(q, k, v, cu, 64, 0.14)
    o.sum().backward(retain_graph=True)
    first, q.grad = q.grad, None
    o.backward(torch.ones_like(o))
    assert torch.equal(first, q.grad)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens,window,post", [([1], 0, True), ([15], 0, True), ([17, 2], 256, True), ([93], 256, True), ([33, 1, 95], 40, False), ([384], 256, True),
                                              ([330, 54], 0, True), ([385], 256, True), ([500, 268], 0, True), ([769], 256, True)])
def test_attention_with_the_output_projection_in_its_launch(dtype, lens, window, post):
    """uvmi_prefill_attn_o at the edges of its 16-token blocks and key tiles, around the 384 and 768 tokens up to which every block's every
    part of 64 and 128 columns has a compute unit, in place, against the attention and a float64 product of what it writes.  Tolerance: the product's rounding to the type, the
    update's, and 512 terms in fp32."""
    import ctypes as C
    from ultraviolet_amd import _lib as L
    from ultraviolet_amd.kernels.gemm import RESID, gemm_args
    from ultraviolet_amd.kernels.varlen_attn import packed_attention, packed_attention_args
    q, k, v, cu = (t.to(DEV) for t in _case(lens, 8, 1, 64, dtype, seed=sum(lens)))
    g = torch.Generator(device=DEV).manual_seed(2)
    N = q.size(0)
    rnd = lambda *s_: torch.randn(*s_, device=DEV, generator=g)
    extra = (torch.nn.functional.normalize(v.float(), dim=-1).contiguous(), rnd(N, 8).sigmoid().contiguous(), rnd(8).tanh().contiguous()) if post else None
    w, x = (rnd(640, 512) / 512 ** 0.5).to(dtype), rnd(N, 640).to(dtype)
    ws = torch.empty(L.lib().uvmi_prefill_attn_workspace_bytes(N), dtype=torch.uint8, device=DEV)
    zg = torch.full((N, 512), 77.0, device=DEV, dtype=dtype)
    y = x.clone()
    a = packed_attention_args(q, k, v, cu, SC, window, zg.view(N, 8, 64), ws, post=extra)
    ga = gemm_args(zg, w, y, RESID, resid=y, ca=0.75, cb=1.25)
    L.check(L.lib().uvmi_prefill_attn_o(C.byref(L.PrefillAttnOArgs(C.addressof(a), C.addressof(ga))), L.stream_ptr(q)), "uvmi_prefill_attn_o")
    assert bool((zg == 77.0).all()) == (N <= 768)
    z = packed_attention(q, k, v, cu, SC, window, post=extra).reshape(N, 512)
    prod = z.double() @ w.double().t()
    want, ulp = 0.75 * x.double() + 1.25 * prod, 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    bound = ulp * (1.25 * prod.abs() + want.abs()) * 1.01 + 512 * 2.0 ** -24 * (z.double().abs() @ w.double().abs().t())
    assert bool(((y.double() - want).abs() <= bound).all()), float(((y.double() - want).abs() / bound).max())
