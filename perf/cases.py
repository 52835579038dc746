"""The calls whose time this repository is measured by.

A case is one forward step, or one hot operation of a step, at a size that a
serving process meets: a shard of a Llama-type or an MLA stack on a batch of
prompt portions or on a replayed decode step (``models``, ``server``), paged
attention over the KV cache, MLA attention over the latent cache, and the
grouped experts (``ops``). Widths are those of the configurations in bench.py
(and of its design comparison for the smaller experts); batches, contexts and
portions range from a single short request to a full batch, and are ragged as
continuous batching makes them. The tensors hold what such steps meet: unit
normal activations, weights of 1/sqrt(fan-in), shuffled cache pages.
"""

import math
import os
import random

import torch

# The first product of a shape picks its library algorithm. Timing the whole
# solution set is for a server's start; here the library's own candidates do.
os.environ.setdefault("PARALLAX_LT_TUNE_FULL", "0")

from parallax_amd import ops  # noqa: E402
from parallax_amd.models import get_model_class  # noqa: E402
from parallax_amd.models.config import ModelConfig  # noqa: E402
from parallax_amd.models.forward_meta import ForwardMeta  # noqa: E402
from parallax_amd.server.graph_runner import DecodeGraphRunner  # noqa: E402
from parallax_amd.server.kv_cache import (  # noqa: E402
    KVCacheSpec, MLAKVCache, PagedKVCache,
)

DEV = "cuda"
PAGE = 32                      # tokens of a cache page in the shard cases
FP8 = torch.float8_e4m3fn
FP8_MAX = 448.0

# The dense stacks of bench.py: width, query heads, key/value heads, head
# width, feed-forward width, vocabulary, layers, bias on q/k/v.
LLAMA = {
    "0.5b": (896, 14, 2, 64, 4864, 151936, 24, True),
    "8b": (4096, 32, 8, 128, 14336, 128256, 32, False),
    "72b": (8192, 64, 8, 128, 29568, 152064, 80, True),
}
# The MLA stack of bench.py (its first, dense layers): width, heads, query
# rank, latent rank, plain / rotated / value head widths, feed-forward width.
MLA = (7168, 128, 1536, 512, 128, 64, 128, 18432, 129280, 61)
# Experts: width, expert width, experts, chosen per token.
EXPERTS = {
    "small": (1024, 512, 16, 2),
    "medium": (2048, 1024, 32, 4),
    "fine": (2048, 768, 128, 8),
    "wide": (7168, 2048, 256, 8),
}
# Attention heads: query heads, key/value heads, head width.
HEADS = {
    "14/2x64": (14, 2, 64),
    "32/8x128": (32, 8, 128),
    "64/8x128": (64, 8, 128),
    "64/8x64": (64, 8, 64),
    "16/16x128": (16, 16, 128),
}


def listed():
    return [
        # Chat with a small model and one user: the shortest step there is,
        # bound by launches and by how fast its weights stream.
        {"name": "llama_decode_one", "kind": "llama_decode", "model": "0.5b",
         "layers": 24, "requests": 1, "longest": 600},
        # A server's decode step at a full ragged batch.
        {"name": "llama_decode_batch", "kind": "llama_decode", "model": "8b",
         "layers": 4, "requests": 96, "longest": 3000},
        # A full prefill step: prompts of unequal length packed to the
        # engine's default chunk.
        {"name": "llama_prefill", "kind": "llama_prefill", "model": "8b",
         "layers": 2, "requests": 3, "tokens": 8192},
        # MLA with W8A8 projections, a decode batch.
        {"name": "mla_layer_decode", "kind": "mla_layer_decode", "fp8": True,
         "requests": 40, "longest": 4000},
        # The same stack on new prompts, bf16.
        {"name": "mla_layer_prefill", "kind": "mla_layer_prefill",
         "fp8": False, "requests": 2, "tokens": 2500},
        # Decode attention alone, as every Llama-type layer calls it.
        {"name": "attention_decode", "kind": "attention_decode",
         "heads": "32/8x128", "requests": 128, "longest": 4096, "page": 32,
         "kv": "bf16", "window": 0, "sinks": False, "softcap": 0.0},
        # Narrow heads, sinks, a quantised cache and odd lengths.
        {"name": "attention_decode_fp8", "kind": "attention_decode",
         "heads": "64/8x64", "requests": 200, "longest": 3001, "page": 16,
         "kv": "fp8", "window": 0, "sinks": True, "softcap": 0.0},
        # The next chunks of two long prompts, on what is cached of them.
        {"name": "attention_prefill_chunk", "kind": "attention_prefill",
         "heads": "32/8x128", "requests": 2, "tokens": 8192, "prefix": 20000,
         "page": 32, "kv": "bf16", "window": 0, "sinks": False,
         "softcap": 0.0},
        # Few very long contexts over the latent cache.
        {"name": "mla_decode_long", "kind": "mla_decode", "heads": 64,
         "requests": 4, "longest": 100000, "kv": "bf16"},
        # Routed experts of a decode step: the weights' stream.
        {"name": "experts_decode", "kind": "experts", "sizes": "fine",
         "tokens": 24, "fp8": False, "limit": 0.0},
        # Routed experts of a prefill step: matrix products.
        {"name": "experts_prefill", "kind": "experts", "sizes": "fine",
         "tokens": 8192, "fp8": False, "limit": 0.0},
        # W8A8 experts of the widest stack, a decode batch.
        {"name": "experts_fp8", "kind": "experts", "sizes": "wide",
         "tokens": 200, "fp8": True, "limit": 0.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["llama_decode", "llama_prefill", "mla_layer_decode",
                       "mla_layer_prefill", "attention_decode",
                       "attention_decode", "attention_prefill",
                       "attention_prefill", "mla_decode", "experts", "experts",
                       "experts"])
    c = {"kind": kind}
    if kind == "llama_decode":
        c["model"] = rng.choice(["0.5b", "8b", "8b", "72b"])
        c["layers"] = {"0.5b": 24, "8b": 4, "72b": 2}[c["model"]]
        c["requests"] = _log(rng, 1, 128)
        c["longest"] = _log(rng, 40, 4000)
    elif kind == "llama_prefill":
        c["model"] = rng.choice(["0.5b", "8b"])
        c["layers"] = 2
        c["requests"] = rng.randint(1, 6)
        c["tokens"] = _log(rng, 60, 8192)
    elif kind == "mla_layer_decode":
        c["fp8"] = rng.random() < 0.5
        c["requests"] = _log(rng, 1, 64)
        c["longest"] = _log(rng, 40, 6000)
    elif kind == "mla_layer_prefill":
        c["fp8"] = rng.random() < 0.5
        c["requests"] = rng.randint(1, 3)
        c["tokens"] = _log(rng, 50, 2500)
    elif kind == "mla_decode":
        c["heads"] = rng.choice([16, 32, 64, 128])
        c["longest"] = _log(rng, 100, 100000)
        c["requests"] = _log(rng, 1, max(1, min(
            256, 400000 * 64 // (c["longest"] * c["heads"]))))
        c["kv"] = rng.choice(["bf16", "bf16", "fp8"])
    elif kind == "experts":
        c["sizes"] = rng.choice(["small", "medium", "fine", "wide"])
        c["fp8"] = c["sizes"] == "wide" or rng.random() < 0.25
        c["tokens"] = _log(rng, 1, 1500 if c["sizes"] == "wide" else 8192)
        c["limit"] = rng.choice([0.0, 0.0, 0.0, 7.0])
    else:
        c["heads"] = rng.choice(sorted(HEADS))
        c["page"] = rng.choice([16, 32, 32, 64])
        c["kv"] = rng.choice(["bf16", "bf16", "fp8"])
        c["window"] = rng.choice([0, 0, 0, 128, 2047])
        c["sinks"] = rng.random() < 0.25
        c["softcap"] = rng.choice([0.0, 0.0, 0.0, 0.0, 30.0])
        if kind == "attention_decode":
            c["longest"] = _log(rng, 40, 32000)
            c["requests"] = _log(rng, 1, max(1, min(512, 600000 // c["longest"])))
        else:
            hq, _, d = HEADS[c["heads"]]
            c["tokens"] = _log(rng, 40, 8192 * 4096 // max(4096, hq * d))
            c["requests"] = rng.randint(1, 6)
            c["prefix"] = rng.choice([0, 0, _log(rng, 100, 20000)])
    return c


# -- sizes that follow from a case (no seed: work() needs them too) -------------


def _lengths(n, longest):
    """Ragged context lengths of n requests, the first one `longest`."""
    r = random.Random(1000003 * n + longest)
    return [longest] + [r.randint(max(1, longest // 4), longest)
                        for _ in range(n - 1)]


def _portions(n, tokens):
    """`tokens` cut into n prompt portions of unequal length."""
    r = random.Random(1000003 * n + tokens)
    n = min(n, tokens)
    cuts = sorted(r.sample(range(1, tokens), n - 1))
    return [b - a for a, b in zip([0] + cuts, cuts + [tokens])]


def _prefixes(n, prefix):
    r = random.Random(7 * n + prefix)
    return [prefix if i == 0 else r.randint(prefix // 2, prefix)
            for i in range(n)]


def _visible(pos, window):
    """Keys a query at position pos sees."""
    return min(pos + 1, window) if window else pos + 1


# -- inputs ------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 2 + 1)


def _randn(g, *shape, scale=1.0, dtype=torch.bfloat16):
    """Normal values, made in slices so that the temporaries stay small."""
    out = torch.empty(*shape, dtype=dtype, device=DEV)
    flat = out.view(-1)
    step = 1 << 27
    for i in range(0, flat.numel(), step):
        part = flat[i:i + step]
        tmp = torch.randn(part.numel(), generator=g, device=DEV,
                          dtype=torch.bfloat16 if dtype == FP8 else dtype)
        part.copy_(tmp.mul_(scale) if scale != 1.0 else tmp)
    return out


def _pages(g, lens, page):
    """Block tables (lists) over a shuffled pool, and the pool's size."""
    counts = [(n + page - 1) // page for n in lens]
    total = sum(counts)
    ids = torch.randperm(total, generator=g, device=DEV).tolist()
    tables, at = [], 0
    for c in counts:
        tables.append(ids[at:at + c])
        at += c
    return tables, total


def _table_tensor(tables):
    width = max(len(t) for t in tables)
    return torch.tensor([t + [0] * (width - len(t)) for t in tables],
                        dtype=torch.int32, device=DEV)


def _slots(table, start, n, page):
    return [table[p // page] * page + p % page for p in range(start, start + n)]


def _int32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def _int64(v):
    return torch.tensor(v, dtype=torch.int64, device=DEV)


def _llama_config(case):
    w, hq, hk, d, ff, vocab, layers, bias = LLAMA[case["model"]]
    return ModelConfig.from_hf_config({
        "architectures": ["Qwen2ForCausalLM" if bias else "LlamaForCausalLM"],
        "model_type": "qwen2" if bias else "llama", "vocab_size": vocab,
        "hidden_size": w, "num_hidden_layers": layers,
        "num_attention_heads": hq, "num_key_value_heads": hk, "head_dim": d,
        "intermediate_size": ff, "rms_norm_eps": 1e-5, "rope_theta": 500000.0,
        "max_position_embeddings": 16384, "qkv_bias": bias,
        "tie_word_embeddings": False, "torch_dtype": "bfloat16",
    })


def _mla_config():
    w, h, qr, r, dn, dr, dv, ff, vocab, layers = MLA
    return ModelConfig.from_hf_config({
        "architectures": ["DeepseekV3ForCausalLM"],
        "model_type": "deepseek_v3", "vocab_size": vocab, "hidden_size": w,
        "num_hidden_layers": layers, "num_attention_heads": h,
        "num_key_value_heads": h, "intermediate_size": ff,
        "moe_intermediate_size": 2048, "n_routed_experts": 256,
        "num_experts_per_tok": 8, "n_shared_experts": 1, "n_group": 8,
        "topk_group": 4, "routed_scaling_factor": 2.5,
        "first_k_dense_replace": 3, "q_lora_rank": qr, "kv_lora_rank": r,
        "qk_nope_head_dim": dn, "qk_rope_head_dim": dr, "v_head_dim": dv,
        "rms_norm_eps": 1e-6, "rope_theta": 10000.0,
        "max_position_embeddings": 16384, "tie_word_embeddings": False,
        "torch_dtype": "bfloat16",
    })


def _llama_weights(case, g):
    """The shard's tensors by parameter name."""
    w, hq, hk, d, ff, vocab, layers, bias = LLAMA[case["model"]]
    out = {"embed_tokens.weight": _randn(g, vocab, w)}
    # a layer adds less than the stream holds, as in a trained stack
    branch = case["layers"] ** -0.5
    for i in range(case["layers"]):
        p = "layers.%d." % i
        n_qkv = (hq + 2 * hk) * d
        out[p + "input_layernorm.weight"] = 1 + _randn(g, w, scale=0.1)
        out[p + "post_attention_layernorm.weight"] = 1 + _randn(g, w, scale=0.1)
        out[p + "self_attn.qkv_proj.weight"] = _randn(g, n_qkv, w, scale=w ** -0.5)
        if bias:
            out[p + "self_attn.qkv_proj.bias"] = _randn(g, n_qkv, scale=0.1)
        out[p + "self_attn.o_proj.weight"] = _randn(
            g, w, hq * d, scale=branch * (hq * d) ** -0.5)
        out[p + "mlp.gate_up_proj.weight"] = _randn(g, 2 * ff, w, scale=w ** -0.5)
        out[p + "mlp.down_proj.weight"] = _randn(g, w, ff,
                                                 scale=branch * ff ** -0.5)
    if case["layers"] == layers:  # a whole stack ends in logits
        out["norm.weight"] = 1 + _randn(g, w, scale=0.1)
        out["lm_head.weight"] = _randn(g, vocab, w, scale=w ** -0.5)
    return out


def _mla_weights(g):
    w, h, qr, r, dn, dr, dv, ff, vocab, _ = MLA
    p = "layers.0."
    a = p + "self_attn."
    return {
        "embed_tokens.weight": _randn(g, vocab, w),
        p + "input_layernorm.weight": 1 + _randn(g, w, scale=0.1),
        p + "post_attention_layernorm.weight": 1 + _randn(g, w, scale=0.1),
        a + "q_a_proj.weight": _randn(g, qr, w, scale=w ** -0.5),
        a + "q_a_layernorm.weight": 1 + _randn(g, qr, scale=0.1),
        a + "q_b_proj.weight": _randn(g, h * (dn + dr), qr, scale=qr ** -0.5),
        a + "kv_a_proj_with_mqa.weight": _randn(g, r + dr, w, scale=w ** -0.5),
        a + "kv_a_layernorm.weight": 1 + _randn(g, r, scale=0.1),
        a + "kv_b_proj.weight": _randn(g, h * (dn + dv), r, scale=r ** -0.5),
        a + "o_proj.weight": _randn(g, w, h * dv, scale=0.5 * (h * dv) ** -0.5),
        p + "mlp.gate_up_proj.weight": _randn(g, 2 * ff, w, scale=w ** -0.5),
        p + "mlp.down_proj.weight": _randn(g, w, ff, scale=0.5 * ff ** -0.5),
    }


def _build(cfg, layers, weights, fp8=False):
    """The shard [0, layers), its parameters replaced by `weights`."""
    with torch.device("meta"):
        model = get_model_class(cfg.architecture)(cfg, 0, layers)
    for name, t in weights.items():
        path, leaf = name.rsplit(".", 1)
        setattr(model.get_submodule(path), leaf,
                torch.nn.Parameter(t, requires_grad=False))
    for m in model.modules():
        for name, b in list(m.named_buffers(recurse=False)):
            if b.device.type == "meta" and name != "rope_cache":
                m.register_buffer(name, torch.empty(
                    b.shape, dtype=torch.bfloat16, device=DEV), persistent=False)
    rot = cfg.qk_rope_head_dim if cfg.is_mla else cfg.rot_dim
    model.rope_cache = _rope_table(cfg.max_position_embeddings, rot,
                                   cfg.rope_theta)
    if hasattr(model, "finalize_weights"):
        model.finalize_weights()
    if fp8:
        for m in list(model.modules()):
            if hasattr(m, "quantize_fp8"):
                m.quantize_fp8()
    return model.eval()


def _rope_table(positions, rot, theta):
    inv = 1.0 / theta ** (torch.arange(0, rot, 2, dtype=torch.float32) / rot)
    f = torch.outer(torch.arange(positions, dtype=torch.float32), inv)
    return torch.cat([f.cos(), f.sin()], dim=-1).to(DEV)


def _shard_inputs(case, seed):
    """Everything of a shard case that has values: weights, token ids, lengths
    before the step, new tokens, pages and the cache's contents."""
    g = _gen(seed)
    mla = case["kind"].startswith("mla")
    if mla:
        weights, vocab, layers = _mla_weights(g), MLA[8], 1
    else:
        weights = _llama_weights(case, g)
        vocab, layers = LLAMA[case["model"]][5], case["layers"]
    if case["kind"].endswith("decode"):
        before = [n - 1 for n in _lengths(case["requests"], case["longest"])]
        new = [1] * len(before)
    else:
        new = _portions(case["requests"], case["tokens"])
        before = [0] * len(new)
    tables, total = _pages(g, [b + n for b, n in zip(before, new)], PAGE)
    ids = torch.randint(0, vocab, (sum(new),), generator=g, device=DEV)
    if mla:
        caches = [_randn(g, total, PAGE, MLA[3] + MLA[5])]
    else:
        _, _, hk, d = LLAMA[case["model"]][:4]
        caches = []
        for _ in range(layers):
            caches.append((_randn(g, total, hk, PAGE, d),
                           _randn(g, total, hk, d, PAGE)))
    return weights, ids, before, new, tables, total, caches


def _prepare_shard(case, seed):
    weights, ids, before, new, tables, total, values = _shard_inputs(case, seed)
    mla = case["kind"].startswith("mla")
    dev = torch.device(DEV)
    if mla:
        cfg = _mla_config()
        model = _build(cfg, 1, weights, case["fp8"])
        cache = MLAKVCache(1, MLA[3], MLA[5], PAGE, 1, dev)
        cache.num_blocks, cache.caches = total, values
        kept = {"cache": values}
    else:
        cfg = _llama_config(case)
        model = _build(cfg, case["layers"], weights)
        cache = PagedKVCache(KVCacheSpec(case["layers"], cfg.num_kv_heads,
                                         cfg.head_dim, PAGE), 1, dev)
        cache.num_blocks = total
        cache.k_caches = [k for k, _ in values]
        cache.v_caches = [v for _, v in values]
        kept = {"k": cache.k_caches, "v": cache.v_caches}
    after = [b + n for b, n in zip(before, new)]
    slots = [s for t, b, n in zip(tables, before, new)
             for s in _slots(t, b, n, PAGE)]
    st = {"kind": case["kind"], "model": model, "kept": kept}
    if case["kind"].endswith("decode"):
        n = len(new)
        st["runner"] = DecodeGraphRunner(
            model, cache, dev, torch.bfloat16, max_batch=n,
            max_model_len=max(1024, (max(after) + 1023) // 1024 * 1024),
            block_size=PAGE, hidden_size=cfg.hidden_size,
            is_first_stage=True, is_last_stage=model.is_last, buckets=[n],
            is_mla=mla)
        st["call"] = dict(input_ids=ids.tolist(), positions=before,
                          slot_mapping=slots, block_tables=tables,
                          seq_lens=after, rids=["r%d" % i for i in range(n)])
        with torch.inference_mode():  # a server captures its graphs up front
            st["runner"].capture_all()
    else:
        st["ids"] = ids
        st["meta"] = ForwardMeta(
            is_prefill=True,
            positions=_int32([p for b, n in zip(before, new)
                              for p in range(b, b + n)]),
            slot_mapping=_int64(slots), block_tables=_table_tensor(tables),
            seq_lens=_int32(after), query_lens=_int32(new),
            kv_cache=None if mla else cache, mla_cache=cache if mla else None,
            logits_indices=_int64([sum(new[:i + 1]) - 1
                                   for i in range(len(new))]),
            max_seq_len=max(after), portions=list(zip(before, new)))
    return st


def _attention_inputs(case, seed):
    g = _gen(seed)
    hq, hk, d = HEADS[case["heads"]]
    if case["kind"] == "attention_decode":
        lens = _lengths(case["requests"], case["longest"])
        new = [1] * len(lens)
    else:
        new = _portions(case["requests"], case["tokens"])
        lens = [n + p for n, p in zip(new, _prefixes(len(new), case["prefix"]))]
    tables, total = _pages(g, lens, case["page"])
    dt = FP8 if case["kv"] == "fp8" else torch.bfloat16
    q = _randn(g, sum(new), hq, d)
    k = _randn(g, total, hk, case["page"], d, dtype=dt)
    v = _randn(g, total, hk, d, case["page"], dtype=dt)
    sinks = torch.randn(hq, generator=g, device=DEV) if case["sinks"] else None
    return q, k, v, tables, lens, new, sinks


def _mla_inputs(case, seed):
    g = _gen(seed)
    lens = _lengths(case["requests"], case["longest"])
    tables, total = _pages(g, lens, PAGE)
    n, h = case["requests"], case["heads"]
    ql = _randn(g, n, h, 512)
    qp = _randn(g, n, h, 64)
    cache = _randn(g, total, PAGE, 576,
                   dtype=FP8 if case["kv"] == "fp8" else torch.bfloat16)
    return ql, qp, cache, tables, lens


def _expert_inputs(case, seed):
    g = _gen(seed)
    H, I, E, k = EXPERTS[case["sizes"]]
    x = _randn(g, case["tokens"], H)
    # experts are not equally popular: a per-expert offset on the logits
    logits = torch.randn(case["tokens"], E, generator=g, device=DEV)
    logits += 0.7 * torch.randn(E, generator=g, device=DEV)
    w, ids = logits.softmax(-1).topk(k, dim=-1)
    w = w / w.sum(-1, keepdim=True)
    if not case["fp8"]:
        gu = _randn(g, E, 2 * I, H, scale=H ** -0.5)
        dn = _randn(g, E, H, I, scale=I ** -0.5)
        return x, ids, w, (gu, None), (dn, None)
    # a normal weight row quantised by its largest value, about 4.4 sigma

    def quantised(rows, cols):
        q = torch.empty(E, rows, cols, dtype=FP8, device=DEV)
        for e in range(E):
            q[e] = torch.randn(rows, cols, generator=g, device=DEV,
                               dtype=torch.bfloat16).mul_(
                FP8_MAX / 4.4).clamp_(-FP8_MAX, FP8_MAX)
        s = 0.9 + 0.2 * torch.rand(E, rows, generator=g, device=DEV)
        return q, s * (4.4 / FP8_MAX * cols ** -0.5)

    return x, ids, w, quantised(2 * I, H), quantised(H, I)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("llama_decode", "llama_prefill", "mla_layer_decode",
                "mla_layer_prefill"):
        return _prepare_shard(case, seed)
    st = {"kind": kind, "case": case}
    if kind in ("attention_decode", "attention_prefill"):
        q, k, v, tables, lens, new, sinks = _attention_inputs(case, seed)
        st["args"] = [q, k, v, _table_tensor(tables), _int32(lens)]
        if kind == "attention_prefill":
            st["args"].append(_int32(new))
        st["args"].append(q.shape[-1] ** -0.5)
        st["kw"] = dict(sliding_window=case["window"] or -1,
                        softcap=case["softcap"], sinks=sinks)
        if kind == "attention_decode":
            st["kw"]["max_seq_len"] = max(lens)
    elif kind == "mla_decode":
        ql, qp, cache, tables, lens = _mla_inputs(case, seed)
        st["args"] = [ql, qp, cache, _table_tensor(tables), _int32(lens),
                      192 ** -0.5]
        st["kw"] = dict(max_seq_len=max(lens))
    else:
        x, ids, w, (gu, gs), (dn, ds) = _expert_inputs(case, seed)
        st["args"] = [x, gu, gs, dn, ds, ids, w] if case["fp8"] \
            else [x, gu, dn, ids, w]
        st["kw"] = dict(limit=case["limit"])
    return st


@torch.inference_mode()
def run(state):
    kind = state["kind"]
    if kind in ("llama_decode", "mla_layer_decode"):
        return {"out": state["runner"].run(**state["call"]), **state["kept"]}
    if kind in ("llama_prefill", "mla_layer_prefill"):
        model = state["model"]
        h = model(model.embed(state["ids"]), state["meta"])
        return {"out": h, **state["kept"]}
    args, kw = state["args"], state["kw"]
    if kind == "attention_decode":
        return ops.paged_attention_decode(*args, **kw)
    if kind == "attention_prefill":
        return ops.prefill_attention(*args, **kw)
    if kind == "mla_decode":
        return ops.mla_paged_attention_decode(*args, **kw)
    if state["case"]["fp8"]:
        return ops.fused_moe_forward_fp8(*args, **kw)
    return ops.fused_moe_forward(*args, **kw)


# -- what a pass cannot do without -----------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("llama_decode", "llama_prefill"):
        w, hq, hk, d, ff, vocab, layers, _ = LLAMA[case["model"]]
        if kind == "llama_decode":
            lens = _lengths(case["requests"], case["longest"])
            T, pairs, ctx = len(lens), sum(lens), sum(lens)
        else:
            new = _portions(case["requests"], case["tokens"])
            T, ctx = sum(new), sum(new)
            pairs = sum(n * (n + 1) // 2 for n in new)
        params = w * (hq + 2 * hk) * d + hq * d * w + 3 * w * ff
        n, head = case["layers"], case["layers"] == layers
        flops = n * (2 * T * params + 4 * pairs * hq * d)
        nbytes = n * (2 * params + 2 * 2 * hk * d * (ctx + T)) + 4 * T * w
        if head:
            flops += 2 * T * w * vocab
            nbytes += 2 * w * vocab + 4 * T * vocab
        return {"bytes": nbytes, "flops": flops}
    if kind in ("mla_layer_decode", "mla_layer_prefill"):
        w, h, qr, r, dn, dr, dv, ff, _, _ = MLA
        size = 1 if case["fp8"] else 2
        plain = w * (qr + r + dr) + h * (dn + dv) * r
        quant = qr * h * (dn + dr) + h * dv * w + 3 * w * ff
        if kind == "mla_layer_decode":
            lens = _lengths(case["requests"], case["longest"])
            T, ctx = len(lens), sum(lens)
            att = 2 * ctx * h * (2 * r + dr)  # absorbed
        else:
            new = _portions(case["requests"], case["tokens"])
            T, ctx = sum(new), sum(new)
            att = sum(n * (n + 1) // 2 for n in new) * h * 2 * (dn + dr + dv)
        return {"bytes": 2 * plain + size * quant + 2 * (r + dr) * (ctx + T)
                + 4 * T * w, "flops": 2 * T * (plain + quant) + att}
    if kind in ("attention_decode", "attention_prefill"):
        hq, hk, d = HEADS[case["heads"]]
        win = case["window"]
        if kind == "attention_decode":
            lens = _lengths(case["requests"], case["longest"])
            T = len(lens)
            read = pairs = sum(_visible(n - 1, win) for n in lens)
        else:
            new = _portions(case["requests"], case["tokens"])
            T, pairs, read = sum(new), 0, 0
            for n, p in zip(new, _prefixes(len(new), case["prefix"])):
                pairs += sum(_visible(p + i, win) for i in range(n))
                read += min(n + p, n + win) if win else n + p
        size = 1 if case["kv"] == "fp8" else 2
        return {"bytes": 2 * size * hk * d * read + 4 * T * hq * d,
                "flops": 4 * pairs * hq * d}
    if kind == "mla_decode":
        ctx = sum(_lengths(case["requests"], case["longest"]))
        n, h = case["requests"], case["heads"]
        size = 1 if case["kv"] == "fp8" else 2
        return {"bytes": size * 576 * ctx + 2 * n * h * (576 + 512),
                "flops": 2 * ctx * h * (576 + 512)}
    H, I, E, k = EXPERTS[case["sizes"]]
    T = case["tokens"]
    # experts that T*k choices touch when the popularity is that of the inputs
    # (a lognormal share of spread 0.7)
    r = random.Random(5)
    share = [math.exp(r.gauss(0.0, 0.7)) for _ in range(E)]
    total = sum(share)
    used = sum(1 - (1 - min(1.0, s / total)) ** (T * k) for s in share)
    return {"bytes": used * 3 * H * I * (1 if case["fp8"] else 2)
            + T * H * (2 + 4) + 12 * T * k, "flops": 6 * T * k * H * I}


def tolerance(case):
    """About four times the error against exact() that was measured (at most
    0.03): results and activations are bf16, so one operation is off by
    1.6e-3 .. 2.3e-3, a stack of layers by the roundings of its stream, W8A8
    by values that round to the neighbouring e4m3 number."""
    if case["kind"].startswith("llama"):
        return {"rel": 0.03 if case["layers"] > 4 else 0.02}
    if case.get("fp8"):
        return {"rel": 0.03}
    return {"rel": 0.012 if case["kind"].startswith("mla_layer") else 0.008}


# -- the same in 64 bits, in plain torch -------------------------------------------


def _rms(x, w, eps):
    return x * (x.pow(2).mean(-1, keepdim=True) + eps).rsqrt() * w.double()


def _quantised(x, dim=None):
    """x rounded to e4m3 with one scale for all of it, or one a row."""
    a = x.abs().amax() if dim is None else x.abs().amax(dim, keepdim=True)
    s = a.clamp_min(1e-8) / FP8_MAX
    return (x / s).clamp(-FP8_MAX, FP8_MAX).float().to(FP8).double() * s


def _product(x, w, fp8=False):
    """x @ w.T; fp8: W8A8 with one scale a tensor."""
    if fp8:
        return _quantised(x) @ _quantised(w.double()).T
    return x @ w.double().T


def _rotated(x, pos, theta, interleaved=False):
    """x: [T, H, D]; halves rotated, or neighbouring pairs."""
    d = x.shape[-1]
    inv = theta ** (-torch.arange(0, d, 2, dtype=torch.float64, device=DEV) / d)
    a = pos.double()[:, None] * inv
    c, s = a.cos()[:, None], a.sin()[:, None]
    if interleaved:
        x1, x2 = x[..., 0::2], x[..., 1::2]
        return torch.stack([x1 * c - x2 * s, x2 * c + x1 * s], -1).flatten(-2)
    x1, x2 = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], -1)


def _attend(q, k, v, scale, first=None, window=0, softcap=0.0, sinks=None):
    """q: [n, Hq, D] at positions first.. (None: all see all keys); k: [L, Hk,
    D]; v: [L, Hk, Dv]. A few rows at a time."""
    n, hq, _ = q.shape
    L, hk = k.shape[:2]
    g = hq // hk
    out = torch.empty(n, hq, v.shape[-1], dtype=torch.float64, device=DEV)
    step = max(1, (1 << 27) // max(1, L * g))
    kpos = torch.arange(L, device=DEV)
    for j in range(hk):
        kj, vj = k[:, j], v[:, j]
        for i in range(0, n, step):
            qi = q[i:i + step, j * g:(j + 1) * g]
            s = (qi.reshape(-1, qi.shape[-1]) @ kj.T).view(*qi.shape[:2], L)
            s *= scale
            if softcap:
                s = softcap * torch.tanh(s / softcap)
            if first is not None:
                pos = (first + i + torch.arange(qi.shape[0], device=DEV))
                hide = kpos[None] > pos[:, None]
                if window:
                    hide |= kpos[None] <= pos[:, None] - window
                s.masked_fill_(hide[:, None], float("-inf"))
            if sinks is not None:
                extra = sinks[j * g:(j + 1) * g].double()
                s = torch.cat([s, extra.view(1, -1, 1).expand(
                    s.shape[0], -1, 1)], -1)
                p = s.softmax(-1)[..., :-1]
            else:
                p = s.softmax(-1)
            out[i:i + step, j * g:(j + 1) * g] = (
                p.reshape(-1, L) @ vj).view(*qi.shape[:2], -1)
    return out


def _paged(cache, table, n, token_dim):
    """The first n tokens of a paged cache, tokens first."""
    pages = cache[torch.tensor(table, device=DEV)]
    if token_dim == 1:          # [pages, tokens, width]
        return pages.flatten(0, 1)[:n].double()
    if token_dim == 3:          # V: [pages, heads, width, tokens]
        pages = pages.transpose(2, 3)
    return pages.transpose(1, 2).flatten(0, 1)[:n].double()


def _exact_llama(case, seed):
    weights, ids, before, new, tables, _, caches = _shard_inputs(case, seed)
    w, hq, hk, d, ff, _, layers, bias = LLAMA[case["model"]]
    eps, theta = 1e-5, 500000.0
    x = weights["embed_tokens.weight"][ids].double()
    pos = _int64([p for b, n in zip(before, new) for p in range(b, b + n)])
    for i in range(case["layers"]):
        p = "layers.%d." % i
        h = _rms(x, weights[p + "input_layernorm.weight"], eps)
        qkv = _product(h, weights[p + "self_attn.qkv_proj.weight"])
        if bias:
            qkv = qkv + weights[p + "self_attn.qkv_proj.bias"].double()
        q, k, v = qkv.split([hq * d, hk * d, hk * d], -1)
        q = _rotated(q.view(-1, hq, d), pos, theta)
        k, v = _rotated(k.view(-1, hk, d), pos, theta), v.view(-1, hk, d)
        att, at = [], 0
        for b, n, t in zip(before, new, tables):
            kk, vv = k[at:at + n], v[at:at + n]
            if b:
                kk = torch.cat([_paged(caches[i][0], t, b, 2), kk])
                vv = torch.cat([_paged(caches[i][1], t, b, 3), vv])
            att.append(_attend(q[at:at + n], kk, vv, d ** -0.5, b))
            at += n
        x = x + _product(torch.cat(att).flatten(1),
                         weights[p + "self_attn.o_proj.weight"])
        h = _rms(x, weights[p + "post_attention_layernorm.weight"], eps)
        a, u = _product(h, weights[p + "mlp.gate_up_proj.weight"]).chunk(2, -1)
        x = x + _product(torch.nn.functional.silu(a) * u,
                         weights[p + "mlp.down_proj.weight"])
    if case["layers"] == layers:
        x = _product(_rms(x, weights["norm.weight"], eps),
                     weights["lm_head.weight"])
    none = [None] * case["layers"]
    return {"out": x, "k": none, "v": none}


def _exact_mla_layer(case, seed):
    weights, ids, before, new, tables, _, caches = _shard_inputs(case, seed)
    w, h, qr, r, dn, dr, dv, ff, _, _ = MLA
    eps, theta, f8 = 1e-6, 10000.0, case["fp8"]
    p = "layers.0."
    a = p + "self_attn."
    x = weights["embed_tokens.weight"][ids].double()
    pos = _int64([q for b, n in zip(before, new) for q in range(b, b + n)])
    y = _rms(x, weights[p + "input_layernorm.weight"], eps)
    q = _rms(_product(y, weights[a + "q_a_proj.weight"]),
             weights[a + "q_a_layernorm.weight"], eps)
    q = _product(q, weights[a + "q_b_proj.weight"], f8).view(-1, h, dn + dr)
    kv = _product(y, weights[a + "kv_a_proj_with_mqa.weight"])
    lat = _rms(kv[:, :r], weights[a + "kv_a_layernorm.weight"], eps)
    kpe = _rotated(kv[:, None, r:], pos, theta, True)[:, 0]
    qpe = _rotated(q[..., dn:], pos, theta, True)
    wkv = weights[a + "kv_b_proj.weight"].double().view(h, dn + dv, r)
    ql = torch.einsum("thd,hdr->thr", q[..., :dn], wkv[:, :dn])
    q = torch.cat([ql, qpe], -1)
    entry = torch.cat([lat, kpe], -1)
    att, at = [], 0
    for b, n, t in zip(before, new, tables):
        e = entry[at:at + n]
        if b:
            e = torch.cat([_paged(caches[0], t, b, 1), e])
        att.append(_attend(q[at:at + n], e[:, None], e[:, None, :r],
                           (dn + dr) ** -0.5, b))
        at += n
    o = torch.einsum("thr,hvr->thv", torch.cat(att), wkv[:, dn:]).flatten(1)
    x = x + _product(o, weights[a + "o_proj.weight"], f8)
    y = _rms(x, weights[p + "post_attention_layernorm.weight"], eps)
    ga, u = _product(y, weights[p + "mlp.gate_up_proj.weight"], f8).chunk(2, -1)
    x = x + _product(torch.nn.functional.silu(ga) * u,
                     weights[p + "mlp.down_proj.weight"], f8)
    return {"out": x, "cache": [None]}


def _exact_attention(case, seed):
    q, k, v, tables, lens, new, sinks = _attention_inputs(case, seed)
    out, at = [], 0
    for t, L, n in zip(tables, lens, new):
        out.append(_attend(q[at:at + n].double(), _paged(k, t, L, 2),
                           _paged(v, t, L, 3), q.shape[-1] ** -0.5, L - n,
                           case["window"], case["softcap"], sinks))
        at += n
    return torch.cat(out)


def _exact_mla(case, seed):
    ql, qp, cache, tables, lens = _mla_inputs(case, seed)
    q = torch.cat([ql, qp], -1).double()
    out = []
    for i, (t, L) in enumerate(zip(tables, lens)):
        e = _paged(cache, t, L, 1)
        out.append(_attend(q[i:i + 1], e[:, None], e[:, None, :512],
                           192 ** -0.5))
    return torch.cat(out)


def _exact_experts(case, seed):
    x, ids, w, (gu, gs), (dn, ds) = _expert_inputs(case, seed)
    I = dn.shape[2]
    xd = x.double()
    if case["fp8"]:
        xd = _quantised(xd, -1)   # activations are quantised a row
    out = torch.zeros(x.shape, dtype=torch.float64, device=DEV)
    for e in range(gu.shape[0]):
        row, col = (ids == e).nonzero(as_tuple=True)
        if not len(row):
            continue
        wg, wd = gu[e].double(), dn[e].double()
        if case["fp8"]:
            wg, wd = wg * gs[e].double()[:, None], wd * ds[e].double()[:, None]
        a = xd[row] @ wg.T
        a, u = a[:, :I], a[:, I:]
        if case["limit"]:
            a = a.clamp(max=case["limit"])
            u = u.clamp(-case["limit"], case["limit"])
            h = (u + 1) * a * torch.sigmoid(1.702 * a)
        else:
            h = torch.nn.functional.silu(a) * u
        if case["fp8"]:
            h = _quantised(h, -1)
        out.index_add_(0, row, (h @ wd.T) * w[row, col].double()[:, None])
    return out


def exact(case, seed):
    with torch.inference_mode():
        kind = case["kind"]
        if kind.startswith("llama"):
            return _exact_llama(case, seed)
        if kind.startswith("mla_layer"):
            return _exact_mla_layer(case, seed)
        if kind.startswith("attention"):
            return _exact_attention(case, seed)
        if kind == "mla_decode":
            return _exact_mla(case, seed)
        return _exact_experts(case, seed)
