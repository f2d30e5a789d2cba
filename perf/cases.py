"""The work that users of this package have it do, as measurable cases on one GPU.

A case is a dict of plain values; `path` names the entry points it goes through:

  decode     patch_model's new_state / decode_step: a caller's own generation loop, one launch sequence per token
  prefill    prefill_packed_host (and prefill for one prompt): prompts into cache rows, logits of their last tokens
  mixed      UVEngine.pack_prompts + mixed_step: prompt chunks and running sequences in one pass
  rollout    Rollout.add / run: continuous batching with captured step graphs until every request is finished
  attention  decode_attention: the ragged decode-attention operator alone
  varlen     varlen_attention and its gradients: packed training sequences
  sample     fused_sample_seeded: softcap, (truncated) draw and log-prob from the head's output

The model is uv-50m-alpha with random weights; token ids, context lengths and prompt lengths are drawn from the seed.
With these weights the next token's logit stands far above the others, so greedy streams do not turn on a last bit."""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from ultraviolet_amd.engine import KVState, UVEngine, UVWeights, make_config, random_params
from ultraviolet_amd.engine.rollout import Rollout
from ultraviolet_amd.kernels import decode_attention, quantize_kv, varlen_attention
from ultraviolet_amd.kernels.fast_decode import patch_model, prefill_packed_host
from ultraviolet_amd.kernels.fused_sample import fused_sample_seeded

DEV = "cuda:0"
CFG = make_config("uv-50m-alpha")
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
HEAD_BYTES = 2 * CFG.vocab_size * CFG.d_model
LAYER_PARAMS = ((CFG.n_heads + 2 * CFG.n_kv_heads) * CFG.head_dim + CFG.n_heads * CFG.head_dim + 3 * CFG.d_ff) * CFG.d_model
TRUNK_PARAMS = CFG.n_layers * LAYER_PARAMS
GLOBAL_LAYERS = sum(CFG.is_global(l) for l in range(CFG.n_layers))
LOCAL_LAYERS = CFG.n_layers - GLOBAL_LAYERS


def listed() -> list[dict]:
    return [
        # one sequence, interactive: the smallest call of a generation loop, where latency counts
        dict(name="decode-1", path="decode", rows=1, lo=200, hi=400, kv="int8", dtype="bf16"),
        # a small odd batch on patch_model's default, the unquantized cache
        dict(name="decode-37-unquantized", path="decode", rows=37, lo=32, hi=700, kv="fp16", dtype="bf16"),
        # the continuous-batching shape: 512 running sequences of 128 .. 2048 tokens
        dict(name="decode-512", path="decode", rows=512, lo=128, hi=2048, kv="int8", dtype="bf16"),
        # one prompt of an interactive session: time to the first token
        dict(name="prefill-1", path="prefill", prompts=1, lo=93, hi=93, kv="int8", dtype="bf16"),
        # a refill of an RL sampler: ragged prompts, packed
        dict(name="prefill-64", path="prefill", prompts=64, lo=64, hi=512, kv="int8", dtype="bf16"),
        # 64 prompt chunks of 512 tokens packed with 448 running sequences
        dict(name="mixed-64x512", path="mixed", prompts=64, length=512, rows=448, lo=256, hi=2048, dtype="bf16"),
        # a small evaluation: short prompts through 16 slots, more requests than slots
        dict(name="rollout-16", path="rollout", slots=16, prompts=24, group=1, lo=16, hi=64, mean_new=40, max_new=64, dtype="bf16"),
        # the GRPO shape: 256 prompts x 8 in 2048 slots, geometric stop lengths
        dict(name="rollout-256x8", path="rollout", slots=2048, prompts=256, group=8, lo=64, hi=256, mean_new=75, max_new=256, dtype="bf16"),
        # the attention operator on an int8 cache, 256 ragged sequences
        dict(name="attention-256", path="attention", rows=256, kv_heads=1, lo=64, hi=1024, kv="int8", dtype="bf16"),
        # ... and on many long sequences, half precision
        dict(name="attention-1000-long", path="attention", rows=1000, kv_heads=1, lo=64, hi=4096, kv="int8", dtype="fp16"),
        # the trainer's packed attention, forward and backward: ragged documents, sliding window
        dict(name="varlen-train", path="varlen", seqs=61, lo=16, hi=1024, window=256, dtype="bf16"),
        # top-k / nucleus sampling of an evaluation batch
        dict(name="sample-200-topk-topp", path="sample", rows=200, top_k=50, top_p=0.95, dtype="bf16"),
    ]


def _logint(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    path = rng.choice(["decode", "prefill", "mixed", "rollout", "attention", "varlen", "sample"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if path == "decode":
        hi = _logint(rng, 64, 2048)
        return dict(path=path, rows=_logint(rng, 1, 1024), lo=max(1, hi // rng.randint(2, 16)), hi=hi, kv=rng.choice(["int8", "int8", "fp16"]), dtype=dtype)
    if path == "prefill":
        hi = _logint(rng, 16, 512)
        return dict(path=path, prompts=_logint(rng, 1, 64), lo=max(1, hi // rng.randint(1, 8)), hi=hi, kv=rng.choice(["int8", "int8", "fp16"]), dtype=dtype)
    if path == "mixed":
        return dict(path=path, prompts=_logint(rng, 1, 64), length=_logint(rng, 16, 512), rows=_logint(rng, 8, 448), lo=64, hi=_logint(rng, 128, 2048), dtype=dtype)
    if path == "rollout":
        slots = _logint(rng, 8, 1024)
        hi, group = _logint(rng, 16, 256), rng.choice([1, 1, 4, 8])
        max_new = _logint(rng, 16, 160)
        return dict(path=path, slots=slots, prompts=max(1, int(slots * rng.uniform(0.5, 1.6)) // group), group=group, lo=max(1, hi // 4), hi=hi,
                    mean_new=max(4, max_new // rng.randint(1, 4)), max_new=max_new, dtype=dtype)
    if path == "attention":
        hi = _logint(rng, 64, 4096)
        kv_heads = rng.choice([1, 1, 2, 8])
        return dict(path=path, rows=_logint(rng, 1, 1024 // kv_heads), kv_heads=kv_heads, lo=max(1, hi // rng.randint(2, 16)), hi=hi,
                    kv=rng.choice(["int8", "int8", "fp16"]), dtype=dtype)
    if path == "varlen":
        hi = _logint(rng, 64, 1024)
        return dict(path=path, seqs=_logint(rng, 1, 61), lo=max(1, hi // rng.randint(1, 64)), hi=hi, window=rng.choice([0, 256]), dtype=dtype)
    top_k, top_p = rng.choice([(0, 1.0), (0, 1.0), (50, 1.0), (0, 0.95), (50, 0.95), (1000, 0.9)])
    return dict(path=path, rows=_logint(rng, 1, 2048 if top_k == 0 and top_p == 1.0 else 512), top_k=top_k, top_p=top_p, dtype=dtype)


# ---------------------------------------------------------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=1)
def _params() -> dict:
    return {k: torch.as_tensor(np.asarray(v), dtype=torch.float32) for k, v in random_params(CFG, 0, perturb=0.02).items()}


class _Model:
    """What patch_model binds to: the configuration and the parameters of a language model, under the reference's names."""

    def __init__(self):
        self.cfg = CFG
        self._parameters_by_name = {k: v.to(DEV) for k, v in _params().items()}

    def state_dict(self):
        return self._parameters_by_name


def _engine(dtype, max_tokens: int) -> UVEngine:
    return UVEngine(UVWeights(CFG, _params(), dtype, DEV), max_tokens)


def _lengths(rng, n: int, lo: int, hi: int) -> np.ndarray:
    """n lengths spread evenly over lo .. hi, in an order of the seed's: the same total whatever the seed."""
    return rng.permutation(np.floor(lo + (hi + 1 - lo) * (np.arange(n) + 0.5) / n).astype(np.int64))


def _new_tokens(n: int, mean: float, most: int) -> np.ndarray:
    """Stop lengths of n requests, geometric with that mean and cut at `most` (at least 2), ascending."""
    q = (np.arange(n) + 0.5) / n
    return np.clip(np.ceil(np.log1p(-q) / np.log1p(-1.0 / mean)), 2, most).astype(np.int64)


def _prompts(rng, lens) -> list:
    return [rng.integers(1, CFG.vocab_size, size=int(n)).tolist() for n in lens]


def _fill_cache(st: KVState, gen: torch.Generator):
    """Contexts already in the cache: values as the quantizer leaves them, or unquantized ones."""
    for l in range(CFG.n_layers):
        for c, sc in ((st.k[l], st.k_scale[l]), (st.v[l], st.v_scale[l])):
            if sc is None:
                c.normal_(generator=gen)
            else:
                c.random_(-127, 128, generator=gen)
                sc.uniform_(0.005, 0.025, generator=gen)


def prepare(case: dict, seed: int) -> dict:
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    path = case["path"]
    if path == "decode":
        rows = case["rows"]
        model = patch_model(_Model(), kv_dtype=case["kv"], dtype=dt, max_tokens=rows)
        st = model.new_state(rows, case["hi"] + 8)
        _fill_cache(st, gen)
        pos = torch.from_numpy(_lengths(rng, rows, case["lo"], case["hi"])).to(DEV)
        toks = [torch.from_numpy(rng.integers(1, CFG.vocab_size, size=rows)).to(DEV) for _ in range(2)]
        return dict(path=path, model=model, st=st, pos=pos, toks=toks)
    if path == "prefill":
        lens = _lengths(rng, case["prompts"], case["lo"], case["hi"])
        model = patch_model(_Model(), kv_dtype=case["kv"], dtype=dt, max_tokens=case["prompts"] * case["hi"])
        prompts = _prompts(rng, lens)
        idx = torch.tensor(prompts, device=DEV) if len(prompts) == 1 else None
        return dict(path=path, model=model, st=model.new_state(len(prompts), case["hi"] + 64), prompts=prompts, idx=idx,
                    starts=torch.zeros(len(prompts), dtype=torch.long, device=DEV), rows=list(range(len(prompts))))
    if path == "mixed":
        n, nd = case["prompts"], case["rows"]
        eng = _engine(dt, n * case["length"] + nd)
        st = KVState(CFG, n + nd, max(case["length"], case["hi"]) + 8, DEV, dtype=dt)
        _fill_cache(st, gen)
        pos = torch.from_numpy(_lengths(rng, nd, case["lo"], case["hi"])).to(DEV)
        return dict(path=path, eng=eng, st=st, pos=pos, starts=torch.zeros_like(pos), rows=torch.arange(nd, device=DEV),
                    tok=torch.from_numpy(rng.integers(1, CFG.vocab_size, size=nd)).to(DEV),
                    prompts=_prompts(rng, [case["length"]] * n), prompt_rows=list(range(nd, nd + n)))
    if path == "rollout":
        eng = _engine(dt, 16384)
        gen_ = Rollout(eng, slots=case["slots"], max_prompt=case["hi"], max_new=case["max_new"], temperature=0.0, bucket=min(128, case["slots"]),
                       share_prompts=case["group"] > 1)
        prompts = [p for p in _prompts(rng, _lengths(rng, case["prompts"], case["lo"], case["hi"])) for _ in range(case["group"])]
        limits = rng.permutation(_new_tokens(len(prompts), case["mean_new"], case["max_new"])).tolist()
        s = dict(path=path, gen=gen_, prompts=prompts, limits=limits)
        run(s)   # a sampler that is already running: its step graphs are captured
        return s
    if path == "attention":
        B, K, hd = case["rows"], case["kv_heads"], CFG.head_dim
        S = (case["hi"] + 31) // 32 * 32
        q = torch.randn(B, CFG.n_heads, hd, device=DEV, generator=gen).to(dt)
        k, v = (torch.randn(B, K, S, hd, device=DEV, generator=gen, dtype=dt) for _ in range(2))
        ks = vs = None
        if case["kv"] == "int8":
            (k, ks), (v, vs) = quantize_kv(k), quantize_kv(v)
        pos = torch.from_numpy(_lengths(rng, B, case["lo"], case["hi"]) - 1).to(DEV)
        return dict(path=path, q=q, k=k, v=v, ks=ks, vs=vs, pos=pos, starts=torch.zeros_like(pos))
    if path == "varlen":
        lens = _lengths(rng, case["seqs"], case["lo"], case["hi"])
        N = int(lens.sum())
        q, go = (torch.randn(1, N, CFG.n_heads, CFG.head_dim, device=DEV, generator=gen, dtype=dt) for _ in range(2))
        k, v = (torch.randn(1, N, CFG.n_kv_heads, CFG.head_dim, device=DEV, generator=gen, dtype=dt) for _ in range(2))
        cu = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).to(DEV)
        return dict(path=path, q=q.requires_grad_(), k=k.requires_grad_(), v=v.requires_grad_(), go=go, cu=cu, longest=int(lens.max()),
                    window=case["window"] or None)
    # the head's output of a trained model: most tokens far down, a few dozen candidates above them
    B, V = case["rows"], CFG.vocab_size
    x = torch.randn(B, V, device=DEV, generator=gen) * 2 - 4
    likely = torch.randint(0, V, (B, 64), device=DEV, generator=gen)
    x.scatter_add_(1, likely, torch.rand(B, 64, device=DEV, generator=gen) * 16)
    return dict(path=path, x=x.to(dt), seed=int(rng.integers(1 << 31)), req=torch.arange(B, device=DEV), top_k=case["top_k"], top_p=case["top_p"],
                tok=torch.from_numpy(rng.integers(0, 512, size=B)).to(DEV))


# ------------------------------------------------------------------------------------------------------------------- run
def run(s: dict):
    path = s["path"]
    if path == "decode":
        # two tokens of the loop: the second attends the first's key; the state goes back to its contexts first
        s["st"].pos.copy_(s["pos"])
        return [s["model"].decode_step(tok, s["st"]) for tok in s["toks"]]
    if path == "prefill":
        if s["idx"] is not None:
            return s["model"].prefill(s["idx"], s["starts"], s["st"]), s["st"].pos
        return prefill_packed_host(s["model"], s["prompts"], s["rows"], s["st"]), s["st"].pos
    if path == "mixed":
        pk = s["eng"].pack_prompts(s["prompts"], s["prompt_rows"], s["st"].max_len, left_pad=False)
        return s["eng"].mixed_step(pk, s["tok"], s["pos"], s["starts"], s["rows"], s["st"])
    if path == "rollout":
        g = s["gen"]
        for i, (p, limit) in enumerate(zip(s["prompts"], s["limits"])):
            g.add(p, i, limit=limit)
        done = sorted(g.run(), key=lambda r: r[0])
        return np.concatenate([np.asarray(r[1], dtype=np.int64) for r in done]), np.concatenate([r[2] for r in done])
    if path == "attention":
        return decode_attention(s["q"], s["k"], s["v"], s["pos"], s["starts"], CFG.attn_scale, k_scale=s["ks"], v_scale=s["vs"])
    if path == "varlen":
        o = varlen_attention(s["q"], s["k"], s["v"], s["cu"], s["longest"], CFG.attn_scale, s["window"])
        return (o, *torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["go"]))
    return fused_sample_seeded(s["x"], s["seed"], s["req"], s["tok"], CFG.softcap, 1.0, top_k=s["top_k"], top_p=s["top_p"])


# ---------------------------------------------------------------------------------------------------- what a pass must do
def _mean_keys(lo: float, hi: float, cap: float = math.inf) -> float:
    """Mean of min(n, cap) for n uniform in lo .. hi."""
    if hi <= cap:
        return (lo + hi) / 2
    if lo >= cap:
        return cap
    inside = (cap - lo) / (hi - lo)
    return inside * (lo + cap) / 2 + (1 - inside) * cap


def _causal_pairs(n: float, window: int) -> float:
    """Query-key pairs of a causal sequence of n tokens."""
    w = min(n, window) if window else n
    return n * w - w * (w - 1) / 2


def _cached_keys(lo: float, hi: float) -> float:
    """Keys a row of context lo .. hi attends, summed over the layers."""
    return GLOBAL_LAYERS * _mean_keys(lo, hi) + LOCAL_LAYERS * _mean_keys(lo, hi, CFG.window)


def work(case: dict) -> dict:
    path, H, hd, d, V = case["path"], CFG.n_heads, CFG.head_dim, CFG.d_model, CFG.vocab_size
    key_bytes = 2 * (hd + 2) if case.get("kv", "int8") == "int8" else 4 * hd
    params = 2 * TRUNK_PARAMS + HEAD_BYTES
    token_flops = 2 * TRUNK_PARAMS
    if path == "decode":
        B, keys = case["rows"], _cached_keys(case["lo"], case["hi"])
        step = {"bytes": params + B * (keys * key_bytes + 4 * V), "flops": B * (token_flops + 2 * d * V + 4 * H * hd * keys)}
        return {k: 2 * v for k, v in step.items()}
    if path == "prefill":
        n, mean = case["prompts"], (case["lo"] + case["hi"]) / 2
        pairs = GLOBAL_LAYERS * _causal_pairs(mean, 0) + LOCAL_LAYERS * _causal_pairs(mean, CFG.window)
        return {"bytes": params + n * mean * (2 * d + CFG.n_layers * key_bytes) + 4 * n * V,
                "flops": n * (mean * token_flops + 2 * d * V + 4 * H * hd * pairs)}
    if path == "mixed":
        n, T, nd, keys = case["prompts"], case["length"], case["rows"], _cached_keys(case["lo"], case["hi"])
        pairs = GLOBAL_LAYERS * _causal_pairs(T, 0) + LOCAL_LAYERS * _causal_pairs(T, CFG.window)
        return {"bytes": 2 * TRUNK_PARAMS + n * T * (2 * d + CFG.n_layers * key_bytes) + nd * keys * key_bytes,
                "flops": (n * T + nd) * token_flops + 4 * H * hd * (n * pairs + nd * keys)}
    if path == "rollout":
        n, mean = case["prompts"] * case["group"], (case["lo"] + case["hi"]) / 2
        new = _new_tokens(n, case["mean_new"], case["max_new"])
        m = float(new.mean())
        # every step reads the weights: the longest request's steps at the least, or all tokens through the slots
        steps = max(int(new.max()), n * m / case["slots"])
        keys = _cached_keys(mean, mean + m)
        unique = case["prompts"] * mean
        return {"bytes": steps * params + n * m * keys * key_bytes + (unique + n * m) * (2 * d + CFG.n_layers * key_bytes),
                "flops": (unique + n * m) * token_flops + n * m * (2 * d * V + 4 * H * hd * keys)}
    if path == "attention":
        B, keys = case["rows"], _mean_keys(case["lo"], case["hi"])
        return {"bytes": B * (case["kv_heads"] * keys * key_bytes + 4 * H * hd + 16), "flops": 4 * H * hd * B * keys}
    if path == "varlen":
        lo, hi = case["lo"], case["hi"]
        lens = _lengths(np.random.default_rng(0), case["seqs"], lo, hi)
        pairs, tokens = sum(_causal_pairs(float(n), case["window"]) for n in lens), float(lens.sum())
        return {"bytes": tokens * hd * 2 * (4 * H + 4 * CFG.n_kv_heads), "flops": 14 * H * hd * pairs}
    return {"bytes": case["rows"] * (2 * V + 28), "flops": 8 * case["rows"] * V}


def tolerance(case: dict):
    """bf16 / fp16 activations with 32-bit accumulation.  Hidden states carry ten layers of such roundings; logits come back
    in 32 bits but are functions of them, flattened by the softcap.  The sampler's sums are 32-bit over 32 768 terms, and
    a draw whose uniform falls on the edge between two tokens may go either way."""
    path, bf16 = case["path"], case["dtype"] == "bf16"
    if path == "sample":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}
    if path == "rollout":
        return {"rel": 5e-3, "max": 0.05, "differ": 0.005}
    if path in ("decode", "prefill"):
        return {"rel": 2e-3, "max": 0.02} if bf16 else {"rel": 5e-4, "max": 5e-3}
    if path == "mixed":
        return {"rel": 2e-2, "max": 0.2} if bf16 else {"rel": 4e-3, "max": 0.04}
    return {"rel": 1e-2, "max": 0.1} if bf16 else {"rel": 3e-3, "max": 0.03}
