"""What this framework is timed on: its KV-cache and attention calls, as programs make them.

Every case goes through a public entry point (the ``flash_attn`` operator namespace, ``KVCache``,
``PhiloxSampler``, the fused pre-attention step, a model's block) on the shapes of the framework's
own workloads: the 12-layer 768-wide quickstart model (12 heads of 64, fp32 or bf16), the
mixed-window stack (12 query / 4 KV heads of 128, window 1024), the decode microbenchmark (32
rows, 16 / 4 heads of 128, up to 8192 keys), the chunked prefill (8 rows, 512-token chunks, 32 / 8
heads of 128) and the large-batch sampling model (d_model 4096, 32 / 8 heads of 128, a 2048-token
prompt shared by 64 rows).

``listed`` gives the named cases, ``draw`` more of the same kinds over the same ranges. Positions
of ragged rows are evenly spaced over [lo, hi] and dealt to the rows by the seed, so that the work
of a case does not depend on it.
"""
from __future__ import annotations

import math

import torch

from modelcore_amd.cache import KVCache
from modelcore_amd.kernels.flash_attn import flash_attn
from modelcore_amd.kernels.qk_epilogue import rope_norm_scale_append
from modelcore_amd.model import ComponentSpec, ModelConfig, ModelManager, rope_tables
from modelcore_amd.runtime import Runtime
from modelcore_amd.sampling import PhiloxSampler

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _device():
    return torch.device("cuda", 0)


# -----------------------------------------------------------------------------------------------
# Cases
# -----------------------------------------------------------------------------------------------
def _attn(name, t_new, batch, heads, kv_heads, dim, dtype, lo, hi, t_max, window=-1, rope=False):
    """An operator call: t_new new tokens per row, appended and attended at positions evenly
    spaced over [lo, hi]. rope: the queries and keys come from a projection and go through the
    fused pre-attention step first, which also appends them."""
    return {"name": name, "kind": "attn", "t_new": t_new, "batch": batch, "heads": heads,
            "kv_heads": kv_heads, "dim": dim, "dtype": dtype, "lo": lo, "hi": hi, "t_max": t_max,
            "window": window, "rope": rope}


def listed():
    return [
        # The smallest call: one token for each of the quickstart's two rows, at the end of its
        # 16-token prompt and 64 new tokens, in its own fp32. All launch latency.
        _attn("quickstart_decode_fp32", 1, 2, 12, 12, 64, "fp32", 79, 79, 80),
        # The quickstart model reading two prompts of its own length in fp32.
        _attn("quickstart_prompt_fp32", 512, 2, 12, 12, 64, "fp32", 0, 0, 576),
        # The quickstart's heads (64 wide, as many KV as query heads) in bf16, serving 16 rows
        # at mixed lengths: the ordinary decode step of a small model.
        _attn("decode_hd64_bf16", 1, 16, 12, 12, 64, "bf16", 128, 2047, 2048),
        # Four whole prompts of such a model, prefilled from an empty cache.
        _attn("prefill_hd64_bf16", 2048, 4, 12, 12, 64, "bf16", 0, 0, 2048),
        # The decode microbenchmark: the largest decode, bound by reading the cache.
        _attn("decode_gqa16x4_8k", 1, 32, 16, 4, 128, "bf16", 512, 8192, 8218),
        # One user's generation after a long prompt: a single row, 16K keys.
        _attn("decode_one_row_16k", 1, 1, 32, 8, 128, "bf16", 16384, 16384, 16896),
        # A chunk in the middle of the chunked prefill of eight 16K prompts, as an attention layer
        # runs it: rope, norm, scale and append in one launch, then the operator.
        _attn("prefill_chunk_gqa32x8", 512, 8, 32, 8, 128, "bf16", 8192, 8192, 16384, rope=True),
        # The next message of one conversation: a hundred new tokens after 8000 cached ones.
        _attn("chat_turn_8k", 100, 1, 32, 8, 128, "bf16", 8000, 8000, 16384),
        # Eight prompts of different lengths prefilled as one packed sequence by the mixed-window
        # stack's local layers (Decoder's multi-prompt prefill).
        {"name": "packed_prompts_w1024", "kind": "packed", "n": 8, "lo": 37, "hi": 4001, "heads": 12,
         "kv_heads": 4, "dim": 128, "dtype": "bf16", "t_max": 4352, "window": 1024},
        # One block of the large-batch sampling model in its captured decode step: 64 rows that
        # share a 2048-token prompt, 200 tokens into their samples.
        {"name": "sampling_block_64", "kind": "block", "batch": 64, "width": 4096, "heads": 32,
         "kv_heads": 8, "hidden": 14336, "prompt": 2048, "done": 200},
        # The draw of the next token of 64 rows from the 50 largest of 32768 logits.
        {"name": "draw_top50_64", "kind": "sample", "batch": 64, "vocab": 32768, "top_k": 50},
        # A 2048-token prompt cache of eight layers replicated into 32 sample rows.
        {"name": "replicate_32_rows", "kind": "replicate", "slots": 8, "rows": 32, "tokens": 2048,
         "kv_heads": 8, "dim": 128, "dtype": "bf16", "t_max": 2560},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# Head groupings (query heads, KV heads) of the framework's workloads and tests.
_HEADS = [(12, 12), (12, 4), (16, 4), (32, 8), (16, 2), (8, 8)]


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 4 + ["packed"] * 2 +
                      ["sample", "sample", "replicate", "block"])
    if kind in ("decode", "prefill", "packed"):
        heads, kv_heads = rng.choice(_HEADS)
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        dim = rng.choice([64, 64, 128, 128, 96, 256])
        window = rng.choice([-1, -1, -1, rng.randint(16, 2048)])
    if kind == "decode":
        hi = _log_int(rng, 48, 16384)
        lo = rng.choice([hi, max(1, hi // 16)])
        # At most the microbenchmark's cache bytes (285 MB) per call.
        row = 2 * hi * kv_heads * dim * (2 if dtype == "bf16" else 4)
        batch = _log_int(rng, 1, max(1, min(64, int(2.8e8 // row))))
        return dict(_attn("", 1, batch, heads, kv_heads, dim, dtype, lo, hi, hi + rng.randint(1, 300),
                          window), name="drawn")
    if kind == "prefill":
        t_new = _log_int(rng, 2, 2048)
        hi = rng.choice([0, _log_int(rng, 16, 8192)])
        lo = rng.choice([hi, hi // 4])
        # The listed cases bound the work: of the widest (64-wide heads, four 2048-token prompts;
        # a chunk of eight 16K prompts on the 128-wide bf16 heads).
        limit = 2.5e10 if dtype == "bf16" else 8e9
        if dtype == "bf16" and dim == 128:
            limit = 2.5e11
        one = 4 * heads * dim * t_new * (hi + t_new / 2)
        while one > limit and t_new > 2:
            t_new //= 2
            one = 4 * heads * dim * t_new * (hi + t_new / 2)
        batch = _log_int(rng, 1, max(1, min(16, int(limit // one))))
        return dict(_attn("", t_new, batch, heads, kv_heads, dim, dtype, lo, hi,
                          hi + t_new + rng.randint(0, 300), window, rng.random() < 0.25),
                    name="drawn")
    if kind == "packed":
        n = rng.randint(2, 12)
        hi = _log_int(rng, 16, 3000 if (dtype == "bf16" and dim == 128) else 700)
        return {"name": "drawn", "kind": "packed", "n": n, "lo": max(1, hi // 8), "hi": hi,
                "heads": heads, "kv_heads": kv_heads, "dim": dim, "dtype": dtype,
                "t_max": hi + rng.randint(0, 300), "window": window}
    if kind == "sample":
        return {"name": "drawn", "kind": "sample", "batch": _log_int(rng, 1, 64),
                "vocab": _log_int(rng, 4096, 131072), "top_k": rng.choice([0, 1, 50, 50, 200, 1000])}
    if kind == "replicate":
        return {"name": "drawn", "kind": "replicate", "slots": rng.randint(1, 12),
                "rows": _log_int(rng, 2, 32), "tokens": _log_int(rng, 16, 1400),
                "kv_heads": rng.choice([4, 8, 12]), "dim": rng.choice([64, 128]),
                "dtype": rng.choice(["bf16", "fp32"]), "t_max": 1500}
    width, heads, kv_heads, hidden = rng.choice([(4096, 32, 8, 14336), (2048, 16, 4, 8192),
                                                 (1536, 12, 4, 4096)])
    return {"name": "drawn", "kind": "block", "batch": _log_int(rng, 1, 64), "width": width,
            "heads": heads, "kv_heads": kv_heads, "hidden": hidden,
            "prompt": _log_int(rng, 32, 2048), "done": rng.randint(1, 400)}


# -----------------------------------------------------------------------------------------------
# Inputs
# -----------------------------------------------------------------------------------------------
def _spread(lo, hi, n):
    return [lo + (hi - lo) * i // (n - 1) for i in range(n)] if n > 1 else [hi]


def _dealt(values, seed):
    order = torch.randperm(len(values), generator=torch.Generator().manual_seed(seed)).tolist()
    return [values[i] for i in order]


def _normal(g, *shape, dtype, scale=1.0):
    return (torch.randn(*shape, generator=g, device=_device()) * scale).to(dtype)


def _filled(g, cache, k_scale=1.2):
    """K rows as the model makes them (RMS-normed, x1.2), V of unit variance."""
    cache.k_cache.normal_(0.0, k_scale, generator=g)
    cache.v_cache.normal_(generator=g)
    return cache


def prepare(case, seed):
    dev = _device()
    g = torch.Generator(device=dev).manual_seed(seed)
    if case["kind"] in ("attn", "packed"):
        dt = DTYPES[case["dtype"]]
        H, Hk, D, T_max = case["heads"], case["kv_heads"], case["dim"], case["t_max"]
    if case["kind"] == "attn":
        B, T = case["batch"], case["t_new"]
        cache = _filled(g, KVCache(B, Hk, T_max, D, 1, dev, dt))
        pos = _dealt(_spread(case["lo"], min(case["hi"], T_max - T), B), seed)
        cache.cache_seqlens.copy_(torch.tensor(pos, dtype=torch.int32))
        s = {"kind": "attn", "cache": cache, "window": (case["window"], 0), "pos": pos,
             "q": _normal(g, B, T, H, D, dtype=dt, scale=1.2),
             "k": _normal(g, B, T, Hk, D, dtype=dt, scale=1.2),
             "v": _normal(g, B, T, Hk, D, dtype=dt)}
        if case["rope"]:
            s["cos"], s["sin"] = rope_tables(T_max, D, dev, dt)
        return s
    if case["kind"] == "packed":
        lens = _dealt(_spread(case["lo"], case["hi"], case["n"]), seed)
        rows = _dealt(list(range(case["n"])), seed + 1)
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        cache = _filled(g, KVCache(case["n"], Hk, T_max, D, 1, dev, dt))
        return {"kind": "packed", "cache": cache, "window": (case["window"], 0), "lens": lens,
                "row_list": rows, "cu": torch.tensor(cu, dtype=torch.int32, device=dev),
                "rows": torch.tensor(rows, dtype=torch.int32, device=dev),
                "q": _normal(g, cu[-1], H, D, dtype=dt, scale=1.2),
                "k": _normal(g, cu[-1], Hk, D, dtype=dt, scale=1.2),
                "v": _normal(g, cu[-1], Hk, D, dtype=dt)}
    if case["kind"] == "sample":
        # Logits under a softcap of 15, as the models' heads give them.
        x = torch.randn(case["batch"], case["vocab"], generator=g, device=dev) * 3.0
        return {"kind": "sample", "logits": 15.0 * torch.tanh(x / 15.0), "top_k": case["top_k"] or None,
                "sampler": PhiloxSampler(case["batch"], dev, base_seed=seed)}
    if case["kind"] == "replicate":
        dt = DTYPES[case["dtype"]]
        src = _filled(g, KVCache(1, case["kv_heads"], case["tokens"], case["dim"], case["slots"],
                                 dev, dt))
        src.advance(case["tokens"])
        dst = KVCache(case["rows"], case["kv_heads"], case["t_max"], case["dim"], case["slots"],
                      dev, dt)
        return {"kind": "replicate", "src": src, "dst": dst}
    return _prepare_block(case, seed, g)


def _block_model(case):
    D = case["width"] // case["heads"]
    block = ComponentSpec("block", {
        "layer_idx": 0, "features": [],
        "mixer": ComponentSpec("attention", {"n_head": case["heads"], "n_kv_head": case["kv_heads"],
                                             "head_dim": D, "window": -1, "kv_slot": None,
                                             "produces_kv": True, "features": []}),
        "ffn": ComponentSpec("gated_mlp", {"activation": "silu", "hidden_dim": case["hidden"]})})
    cfg = ModelConfig(sequence_len=case["prompt"] + case["done"] + 64, vocab_size=256,
                      n_embd=case["width"],
                      shared={"rope": ComponentSpec("rotary", {"head_dim": D, "over_compute": 1}),
                              "norm": ComponentSpec("rms_norm", {"eps": None})},
                      input=ComponentSpec("token_embedding", {"smear": False}),
                      body=ComponentSpec("stack", {"blocks": [block], "features": []}),
                      output=ComponentSpec("lm_head", {"softcap": 15}))
    mgr = ModelManager(Runtime(torch.bfloat16))
    return mgr, cfg


def _prepare_block(case, seed, g):
    """A block with cached bf16 weights on the decode products, its cache (a shared prompt, then
    each row's own tokens) and the captured graph of its decode step."""
    dev = _device()
    mgr, cfg = _block_model(case)
    model = mgr.create_model(cfg, device=dev, seed=seed)
    block = model.body.blocks[0]
    with torch.no_grad():  # the projections that init leaves at zero, as in a trained model
        for w in (block.mixer.c_proj.weight, block.ffn.down_proj.weight):
            w.normal_(0.0, w.shape[1] ** -0.5, generator=g)
    model.cache_inference_weights()
    model.use_skinny_gemm(True)
    model.set_fused_residual(True)
    P, n = case["prompt"], case["done"]
    cache = mgr.new_kv_cache(model, batch_size=case["batch"], seq_len=P + n + 64)
    prompt = _filled(g, mgr.new_kv_cache(model, batch_size=1, seq_len=P))
    prompt.advance(P)
    cache.prefill(prompt)
    cache.k_cache[:, :, P:].normal_(0.0, 1.2, generator=g)
    cache.v_cache[:, :, P:].normal_(generator=g)
    cache.advance(n)
    x = _normal(g, case["batch"], 1, case["width"], dtype=torch.bfloat16)
    s = {"kind": "block", "block": block, "cache": cache, "x": x, "model": model}

    def step():
        return block.forward_carry(x, None, cache, {})

    with torch.inference_mode():
        side = torch.cuda.Stream(device=dev)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"], stream=side):
            s["out"] = step()
        torch.cuda.current_stream().wait_stream(side)
    return s


# -----------------------------------------------------------------------------------------------
# One pass
# -----------------------------------------------------------------------------------------------
def run(s):
    if s["kind"] == "attn":
        cache = s["cache"]
        kc, vc = cache.get_slot_cache(0)
        q, k, v = s["q"], s["k"], s["v"]
        if "cos" in s:
            q = rope_norm_scale_append(q, s["cos"], s["sin"], cache.cache_seqlens, k, v, kc, vc)
            k = v = None
        y = flash_attn.flash_attn_with_kvcache(q, kc, vc, k=k, v=v,
                                               cache_seqlens=cache.cache_seqlens, causal=True,
                                               window_size=s["window"])
        return [y, kc, vc]
    if s["kind"] == "packed":
        kc, vc = s["cache"].get_slot_cache(0)
        y = flash_attn.flash_attn_varlen_with_kvcache(
            s["q"], kc, vc, k=s["k"], v=s["v"], cache_seqlens=s["cache"].cache_seqlens,
            cu_seqlens=s["cu"], max_seqlen=max(s["lens"]), rows=s["rows"], causal=True,
            window_size=s["window"])
        return [y, kc, vc]
    if s["kind"] == "sample":
        return [s["sampler"](s["logits"], 1.0, s["top_k"]), s["sampler"].offsets]
    if s["kind"] == "replicate":
        s["dst"].reset()
        s["dst"].prefill(s["src"])
        return [s["dst"].k_cache, s["dst"].v_cache, s["dst"].cache_seqlens]
    s["graph"].replay()
    kc, vc = s["cache"].get_slot_cache(0)
    return [*s["out"], kc, vc]


# -----------------------------------------------------------------------------------------------
# What a pass cannot do without
# -----------------------------------------------------------------------------------------------
def _pairs(pos, T, window):
    """(query, key) pairs of T tokens from position pos on, and the keys they read in all."""
    if window < 0:
        return T * pos + T * (T + 1) // 2, pos + T
    full = max(0, min(T, window - pos + 1))  # queries that still see key 0
    pairs = full * pos + full * (full + 1) // 2 + (T - full) * (window + 1)
    return pairs, pos + T - max(0, pos - window)


def work(case):
    if case["kind"] in ("attn", "packed"):
        H, Hk, D = case["heads"], case["kv_heads"], case["dim"]
        size = 2 if case["dtype"] == "bf16" else 4
        if case["kind"] == "attn":
            seqs = [(p, case["t_new"]) for p in
                    _spread(case["lo"], min(case["hi"], case["t_max"] - case["t_new"]), case["batch"])]
        else:
            seqs = [(0, n) for n in _spread(case["lo"], case["hi"], case["n"])]
        total = sum(t for _, t in seqs)
        seen = [_pairs(p, t, case["window"]) for p, t in seqs]
        old = sum(keys for _, keys in seen) - total  # cached keys read; the new ones come as k, v
        rows = 2 * total * H * D + 2 * Hk * D * (old + 2 * total)  # q, out; K/V read, new ones written
        return {"bytes": rows * size, "flops": 4 * H * D * sum(p for p, _ in seen)}
    if case["kind"] == "sample":
        return {"bytes": case["batch"] * case["vocab"] * 4, "flops": 0}
    if case["kind"] == "replicate":
        size = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": 2 * case["slots"] * case["tokens"] * case["kv_heads"] * case["dim"] * size *
                (case["rows"] + 1), "flops": 0}
    B, W, H, Hk, F = case["batch"], case["width"], case["heads"], case["kv_heads"], case["hidden"]
    D = W // H
    weights = W * (H + 2 * Hk) * D + H * D * W + 3 * W * F
    keys = case["prompt"] + B * (case["done"] + 1)
    return {"bytes": 2 * (weights + 2 * keys * Hk * D + 3 * B * W),
            "flops": 2 * B * weights + 4 * H * D * B * (case["prompt"] + case["done"] + 1)}


def tolerance(case):
    if case["kind"] in ("sample", "replicate"):
        return "exact"
    if case["kind"] == "block":
        return {"rel": 1e-2, "max": 0.2}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 1e-5, "max": 1e-4}


# -----------------------------------------------------------------------------------------------
# The same in 64 bits
# -----------------------------------------------------------------------------------------------
def _attend(q, kc, vc, pos, window, scale):
    """q (T, H, D) from position pos on, against one row's kc, vc (T_max, H_kv, D); 64 bits."""
    T, H, D = q.shape
    Hk = kc.shape[1]
    G = H // Hk
    L = pos + T
    lo = max(0, pos - window) if window >= 0 else 0
    rows = torch.arange(pos, L, device=q.device)[:, None]
    cols = torch.arange(lo, L, device=q.device)[None, :]
    hidden = cols > rows
    if window >= 0:
        hidden = hidden | (rows - cols > window)
    out = torch.empty_like(q)
    for h in range(H):
        k = kc[lo:L, h // G].contiguous()
        s = (q[:, h].contiguous() @ k.t().contiguous()) * scale
        s.masked_fill_(hidden, float("-inf"))
        out[:, h] = torch.softmax(s, dim=-1) @ vc[lo:L, h // G].contiguous()
    return out


def _rope_norm(x, cos, sin, pos, scale=1.2):
    """x (T, heads, D) rotated at positions pos.., RMS-normed and scaled; 64 bits."""
    T, half = x.shape[0], x.shape[-1] // 2
    c, s = cos[pos:pos + T, None], sin[pos:pos + T, None]
    a, b = x[..., :half], x[..., half:]
    r = torch.cat([a * c + b * s, b * c - a * s], -1)
    eps = torch.finfo(torch.float32).eps
    return r / torch.sqrt(r.square().mean(-1, keepdim=True) + eps) * scale


def exact(case, seed):
    if case["kind"] in ("sample", "replicate"):
        return None
    s = prepare(case, seed)
    kc, vc = (t.double() for t in s["cache"].get_slot_cache(0))
    if case["kind"] == "block":
        return _exact_block(case, s, kc, vc)
    q, k, v = s["q"].double(), s["k"].double(), s["v"].double()
    scale = case["dim"] ** -0.5
    out = torch.empty_like(q)
    if case["kind"] == "attn":
        for b, pos in enumerate(s["pos"]):
            qb, kb = q[b], k[b]
            if case["rope"]:
                cos, sin = s["cos"][0, :, 0].double(), s["sin"][0, :, 0].double()
                qb, kb = _rope_norm(qb, cos, sin, pos), _rope_norm(kb, cos, sin, pos)
            T = qb.shape[0]
            kc[b, pos:pos + T], vc[b, pos:pos + T] = kb, v[b]
            out[b] = _attend(qb, kc[b], vc[b], pos, case["window"], scale)
        return [out, kc, vc]
    at = 0
    for n, row in zip(s["lens"], s["row_list"]):
        kc[row, :n], vc[row, :n] = k[at:at + n], v[at:at + n]
        out[at:at + n] = _attend(q[at:at + n], kc[row], vc[row], 0, case["window"], scale)
        at += n
    return [out, kc, vc]


def _exact_block(case, s, kc, vc):
    m, f = s["block"].mixer, s["block"].ffn
    H, Hk = case["heads"], case["kv_heads"]
    D = case["width"] // H
    eps = torch.finfo(torch.float32).eps
    norm = lambda t: t / torch.sqrt(t.square().mean(-1, keepdim=True) + eps)  # noqa: E731
    w = lambda lin: lin.weight.to(torch.bfloat16).double().t().contiguous()  # noqa: E731
    x = s["x"][:, 0].double()
    h = norm(x)
    pos = case["prompt"] + case["done"]
    cos, sin = m.rope.cos[0, :, 0].double(), m.rope.sin[0, :, 0].double()
    q = (h @ w(m.c_q)).view(-1, H, D)
    k = (h @ w(m.c_k)).view(-1, Hk, D)
    v = (h @ w(m.c_v)).view(-1, Hk, D)
    y = torch.empty_like(q)
    for b in range(case["batch"]):
        kc[b, pos:pos + 1] = _rope_norm(k[b:b + 1], cos, sin, pos)
        vc[b, pos:pos + 1] = v[b:b + 1]
        y[b:b + 1] = _attend(_rope_norm(q[b:b + 1], cos, sin, pos), kc[b], vc[b], pos, -1,
                             D ** -0.5)
    x = x + y.flatten(1) @ w(m.c_proj)
    h = norm(x)
    gate = h @ w(f.gate_proj)
    x = x + (gate * torch.sigmoid(gate) * (h @ w(f.up_proj))) @ w(f.down_proj)
    return [x[:, None], norm(x)[:, None], kc, vc]
