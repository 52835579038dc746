"""Products of few rows whose parts are added up and normed in one launch: the same bits
as product, residual, norm and conversion apart; layers that take it against the same
layers with a hook, which do not."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from parallax_amd import ops
from parallax_amd.models.forward_meta import ForwardMeta


def _rand(g, *s):
    return torch.randn(*s, generator=g, device="cuda").bfloat16()


def _fp8(w):
    scale = (w.float().abs().amax() / 448).reshape(1)
    return (w.float() / scale).clamp(-448, 448).to(torch.float8_e4m3fn), scale


@pytest.mark.parametrize("M,N,K,fp8", [
    (40, 1536, 7168, False), (33, 4096, 4096, False), (64, 8192, 7168, False),
    (17, 1032, 6144, False), (32, 4096, 14336, False), (128, 8192, 8192, False),
    (40, 7168, 16384, True), (97, 7168, 18432, True),
    (34, 520, 7168, False),
])
@pytest.mark.parametrize("quantize", [False, True])
def test_linear_norm_is_the_launches_apart(M, N, K, fp8, quantize):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, w = _rand(g, M, K), _rand(g, N, K) * K ** -0.5
    norm, res = 1 + 0.1 * _rand(g, N), (_rand(g, M, N + 8) * 3)[:, :N]
    scale = None
    if fp8:
        w, scale = _fp8(w)
    p = ops.linear_fp8(x, w, scale) if fp8 else ops.linear(x, w)
    for residual in (None, res):
        got = ops.linear_norm(x, w, scale, residual, norm, 1e-6, quantize)
        assert got is not None
        if residual is None:
            want, sums = ops.rmsnorm(p, norm, 1e-6), None
        else:
            want, sums = ops.fused_add_rmsnorm(p.clone(), residual.contiguous().clone(),
                                               norm, 1e-6)
        if quantize:
            q, s = ops._require_ext("t").quantize_fp8_tensor(want)
            assert torch.equal(got[0].view(torch.uint8), q.view(torch.uint8))
            assert torch.equal(got[1], s)
        else:
            assert got[1] is None and torch.equal(got[0], want)
        assert sums is None and got[2] is None or torch.equal(got[2], sums)


def test_linear_norm_infinities():
    """Where a row's sums are infinite or cancel so, the launches apart say the same, and
    the other rows are finite. (40 rows, as above.)"""
    g = torch.Generator(device="cuda").manual_seed(3)
    x, w = _rand(g, 40, 7168), _rand(g, 1536, 7168) * 7168 ** -0.5
    norm, res = 1 + 0.1 * _rand(g, 1536), _rand(g, 40, 1536)
    x[3, 7167] = x[20, 0] = float("inf")
    res[20, 100] = res[39, 1535] = float("-inf")
    got = ops.linear_norm(x, w, None, res, norm, 1e-6)
    want = ops.fused_add_rmsnorm(ops.linear(x, w), res.clone(), norm, 1e-6)
    for a, b in ((got[0], want[0]), (got[2], want[1])):
        torch.testing.assert_close(a, b, rtol=0, atol=0, equal_nan=True)
        assert (~a.isfinite()).any(1).nonzero()[:, 0].tolist() == [3, 20, 39]


def test_linear_norm_without_a_kernel():
    g = torch.Generator(device="cuda").manual_seed(0)
    x, w, n = _rand(g, 40, 4096), _rand(g, 4096, 4096), _rand(g, 4096)
    call = lambda x=x, w=w, r=None, n=n: ops.linear_norm(x, w, None, r, n, 1e-5)
    assert call() is not None
    assert call(x=x[:4]) is None and call(x=x[:0]) is None
    wq, scale = _fp8(_rand(g, 7168, 16384))                  # 9 rows: without parts
    assert ops.linear_norm(_rand(g, 9, 16384), wq, scale, None, _rand(g, 7168), 1e-5) is None
    assert call(x=x.float()) is None and call(w=w.float()) is None
    assert call(x=_rand(g, 40, 4100)[:, 4:]) is None         # rows at odd places
    assert call(n=n[:4088]) is None and call(r=_rand(g, 39, 4096)) is None
    assert call(x=_rand(g, 129, 4096)) is None
    assert call(w=w.clone().requires_grad_()) is None


@pytest.mark.parametrize("T,I", [(1, 8), (3, 136), (40, 18432), (128, 1000)])
def test_silu_and_mul_fp8(T, I):
    g = torch.Generator(device="cuda").manual_seed(I)
    x = _rand(g, T, 2 * I)
    q, s = ops.silu_and_mul_fp8(x)
    q2, s2 = ops._require_ext("t").quantize_fp8_tensor(ops.silu_and_mul(x))
    assert torch.equal(q.view(torch.uint8), q2.view(torch.uint8)) and torch.equal(s, s2)


WIDTH = 7168  # products of these widths have parts, in fp8 too


def _layer(kind, fp8):
    from parallax_amd.models.config import ModelConfig
    kw = dict(vocab_size=64, hidden_size=WIDTH, num_layers=1, num_heads=56,
              num_kv_heads=4, head_dim=128, intermediate_size=512,
              max_position_embeddings=256, eos_token_ids=[])
    if kind == "mla":
        from parallax_amd.models.deepseek_v3 import DeepseekV3DecoderLayer as Layer
        kw.update(q_lora_rank=1536, kv_lora_rank=512, qk_nope_head_dim=128,
                  qk_rope_head_dim=64, v_head_dim=128, num_kv_heads=56)
    else:
        from parallax_amd.models.llama import LlamaDecoderLayer as Layer
    cfg = ModelConfig(architecture="x", **kw)
    with torch.device("cuda"):
        layer = Layer(cfg, 0, 0).to(torch.bfloat16).eval()
    g = torch.Generator(device="cuda").manual_seed(1)
    for name, p in layer.named_parameters():
        p.data.copy_(1 + 0.1 * torch.randn(p.shape, generator=g, device="cuda")
                     if p.dim() == 1 else
                     torch.randn(p.shape, generator=g, device="cuda") * p.shape[1] ** -0.5)
    if kind == "mla":
        layer.self_attn.finalize_weights()
    if fp8:
        for m in list(layer.modules()):
            if hasattr(m, "quantize_fp8"):
                m.quantize_fp8()
    return layer


def _step(layer, kind, T, first=False, change=lambda t: t):
    from parallax_amd.server.kv_cache import KVCacheSpec, MLAKVCache, PagedKVCache
    dev = torch.device("cuda")
    g = torch.Generator(device="cuda").manual_seed(T)
    if kind == "mla":
        cache = MLAKVCache(1, 512, 64, 16, T, dev)
        kept = cache.caches
    else:
        cache = PagedKVCache(KVCacheSpec(1, 4, 128, 16), T, dev)
        kept = cache.k_caches + cache.v_caches
    for c in kept:
        c.copy_(torch.randn(c.shape, generator=g, device="cuda"))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    lens = [1 + i % 16 for i in range(T)]
    meta = ForwardMeta(
        is_prefill=False, positions=i32([n - 1 for n in lens]),
        slot_mapping=torch.tensor([16 * i + n - 1 for i, n in enumerate(lens)],
                                  device=dev),
        block_tables=i32([[i] for i in range(T)]), seq_lens=i32(lens),
        kv_cache=None if kind == "mla" else cache,
        mla_cache=cache if kind == "mla" else None, max_seq_len=16, appends=True)
    rope = torch.randn(32, 64 if kind == "mla" else 128, generator=g, device="cuda")
    x, res = _rand(g, T, WIDTH), change(_rand(g, T, WIDTH))
    with torch.inference_mode():
        out = layer(res, None, meta, rope) if first else layer(x, res, meta, rope)
        return list(out) + list(kept)


@pytest.mark.parametrize("kind,fp8", [("llama", False), ("llama", True), ("mla", False),
                                      ("mla", True)])
@pytest.mark.parametrize("T", [1, 40, 128])
def test_a_hook_sees_the_product_and_changes_nothing(kind, fp8, T, monkeypatch):
    """The joined launches run where nothing looks on, with the scales of fp8 layers, and
    not where hooks do: the same bits either way."""
    joined = []
    linear_norm = ops.linear_norm

    def spy(x, w, scale, residual, norm, eps, quantize=False):
        out = linear_norm(x, w, scale, residual, norm, eps, quantize)
        joined.append((w.shape[0], quantize, out is not None))
        return out

    monkeypatch.setattr(ops, "linear_norm", spy)
    layer = _layer(kind, fp8)
    want = _step(layer, kind, T)
    assert joined == ([] if T == 1 else
                      [(1536, fp8, True)] * (kind == "mla") + [(WIDTH, fp8, True)])
    joined.clear()
    seen = []
    layer.self_attn.o_proj.register_forward_hook(lambda m, a, out: seen.append(out.shape))
    layer.post_attention_layernorm.register_forward_hook(
        lambda m, a, out: seen.append(out[0].shape))
    if kind == "mla":
        layer.self_attn.q_a_layernorm.register_forward_hook(
            lambda m, a, out: seen.append(out.shape))
    got = _step(layer, kind, T)
    assert len(seen) == (3 if kind == "mla" else 2) and not joined
    assert all(torch.equal(a, b) for a, b in zip(got, want))



@pytest.mark.parametrize("kind", ["llama", "mla"])
@pytest.mark.parametrize("T", [2, 4, 40, 130])
@pytest.mark.parametrize("first", [False, True])
def test_a_residual_of_rows_apart_is_refused(kind, T, first):
    """As the norm that adds it refuses it, of any number of rows: it adds in place.
    first: a stack's first layer, whose input is the residual."""
    layer = _layer(kind, False)
    with pytest.raises(RuntimeError, match="contiguous"):
        _step(layer, kind, T, first, lambda t: torch.cat([t, t], 1)[:, :WIDTH])


def _shard(kind, fp8, last, experts=0):
    from parallax_amd.models import get_model_class
    from parallax_amd.models.config import ModelConfig
    kw = dict(vocab_size=64, hidden_size=WIDTH, num_layers=3, num_heads=56,
              num_kv_heads=4, head_dim=128, intermediate_size=4096,
              max_position_embeddings=256, eos_token_ids=[])
    if kind == "mla":
        kw.update(q_lora_rank=1536, kv_lora_rank=512, qk_nope_head_dim=128,
                  qk_rope_head_dim=64, v_head_dim=128, num_kv_heads=56)
    if experts:  # but for the first layer
        kw.update(num_experts=experts, num_experts_per_tok=2, moe_intermediate_size=64,
                  first_k_dense_layers=1)
    name = "DeepseekV3ForCausalLM" if kind == "mla" else "LlamaForCausalLM"
    with torch.device("cuda"):
        model = get_model_class(name)(ModelConfig(architecture=name, **kw), 0,
                                      3 if last else 2).to(torch.bfloat16).eval()
    g = torch.Generator(device="cuda").manual_seed(1)
    for p in model.parameters():
        p.data.copy_(1 + 0.1 * torch.randn(p.shape, generator=g, device="cuda")
                     if p.dim() == 1 else
                     torch.randn(p.shape, generator=g, device="cuda") * p.shape[1] ** -0.5)
    model.rope_cache = model.rope_cache.float()
    if kind == "mla":
        model.finalize_weights()
    if fp8:
        for layer in model.layers:
            for m in list(layer.modules()):
                if hasattr(m, "quantize_fp8"):
                    m.quantize_fp8()
    return model


def _shard_step(model, kind, T):
    """One decode step of T requests: what the model returns, and its caches."""
    from parallax_amd.server.kv_cache import KVCacheSpec, MLAKVCache, PagedKVCache
    dev = torch.device("cuda")
    n = len(model.layers)
    g = torch.Generator(device="cuda").manual_seed(T)
    if kind == "mla":
        cache = MLAKVCache(n, 512, 64, 16, T, dev)
        kept = cache.caches
    else:
        cache = PagedKVCache(KVCacheSpec(n, 4, 128, 16), T, dev)
        kept = cache.k_caches + cache.v_caches
    for c in kept:
        c.copy_(torch.randn(c.shape, generator=g, device="cuda"))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    lens = [1 + i % 16 for i in range(T)]
    meta = ForwardMeta(
        is_prefill=False, positions=i32([n - 1 for n in lens]),
        slot_mapping=torch.tensor([16 * i + n - 1 for i, n in enumerate(lens)],
                                  device=dev),
        block_tables=i32([[i] for i in range(T)]), seq_lens=i32(lens),
        kv_cache=None if kind == "mla" else cache,
        mla_cache=cache if kind == "mla" else None, max_seq_len=16, appends=True)
    with torch.inference_mode():
        return [model(_rand(g, T, WIDTH), meta)] + list(kept)


@pytest.mark.parametrize("kind,fp8", [("llama", False), ("llama", True), ("mla", False),
                                      ("mla", True)])
@pytest.mark.parametrize("last", [False, True])
def test_layers_that_end_in_the_next_norm(kind, fp8, last, monkeypatch):
    """The parts of an MLP's last product are added up by the next layer's norm, the
    shard's norm or its last sum, and by a launch of their own where a hook looks on: the
    same bits either way."""
    model = _shard(kind, fp8, last)
    n = len(model.layers)
    step = lambda T: _shard_step(model, kind, T)
    calls = []
    for name in ("linear_norm", "linear_add"):
        def spy(x, w, *args, of=getattr(ops, name), name=name, **kw):
            out = of(x, w, *args, **kw)
            if w.shape[1] == 4096 and out is not None:  # a down projection
                calls.append(name)
            return out
        monkeypatch.setattr(ops, name, spy)
    rows = (4, 5, 33, 128, 130)
    want = [step(T) for T in rows]
    # five rows' products have no parts, of more than 128 none has
    few = [T for T in rows if ops.product_has_parts(
        T, next(iter(model.layers)).mlp.down_proj.weight_fp8 if fp8
        else next(iter(model.layers)).mlp.down_proj.weight)]
    assert 33 in few and 4 not in few and 130 not in few
    assert calls == (["linear_norm"] * (n - 1) + ["linear_norm" if last else "linear_add"]
                     ) * len(few)
    calls.clear()
    for layer in model.layers:
        layer.register_forward_hook(lambda m, a, out: None)
    for T, w in zip(rows, want):
        assert all(torch.equal(a, b) for a, b in zip(w, step(T))), T
    assert not calls


@pytest.mark.parametrize("kind,where", [
    (kind, where) for kind in ("llama", "mla")
    for where in ("mlp", "layer", "input_layernorm", "experts", "no kernel")
    if kind == "mla" or where != "experts"])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("last", [False, True])
def test_layers_of_which_one_does_not_end_so(kind, fp8, where, last, monkeypatch):
    """A layer that gets its input normed and does not end in the next norm, one behind a
    layer that may not, and products left to the caller behind an opened MLP: the bits of
    the layers one by one."""
    T = 33
    model = _shard(kind, fp8, last, experts=4 if where == "experts" else 0)
    joined = []
    for name in ("linear_norm", "linear_add"):
        def spy(x, w, *args, of=getattr(ops, name), name=name, **kw):
            if w.shape[1] != 4096:
                return of(x, w, *args, **kw)
            joined.append(name)
            return None if where == "no kernel" else of(x, w, *args, **kw)
        monkeypatch.setattr(ops, name, spy)
    if where in ("mlp", "layer", "input_layernorm"):
        at = model.layers[1]
        (at if where == "layer" else getattr(at, where)).register_forward_hook(
            lambda m, a, out: None)
    got = _shard_step(model, kind, T)
    norm, add = "linear_norm", "linear_add"
    assert joined == (  # of three layers and the last norm, or of two and a sum
        {"mlp": [norm, norm], "layer": [norm], "input_layernorm": [norm, norm],
         "experts": [norm], "no kernel": [norm, norm, norm]} if last else
        {"mlp": [norm], "layer": [], "input_layernorm": [add], "experts": [norm],
         "no kernel": [norm, add]})[where]
    joined.clear()
    for layer in model.layers:
        layer.register_forward_hook(lambda m, a, out: None)
    want = _shard_step(model, kind, T)
    assert not joined and all(torch.equal(a, b) for a, b in zip(got, want))
    assert got[0].isfinite().all()


@pytest.mark.parametrize("M,N,K", [(9, 7168, 16384), (33, 4096, 4096), (128, 8192, 8192)])
@pytest.mark.parametrize("fp8", [False, True])
def test_linear_add(M, N, K, fp8):
    """The bits of the product and the sum apart; rows of a residual that lie apart."""
    g = torch.Generator(device="cuda").manual_seed(M)
    x, w = _rand(g, M, K), _rand(g, N, K) * K ** -0.5
    res = _rand(g, M, N + 8)[:, :N]
    scale = None
    if fp8:
        scale = (w.float().abs().amax() / 448).reshape(1)
        w = (w.float() / scale).to(torch.float8_e4m3fn)
    if not ops.product_has_parts(M, w):
        assert ops.linear_add(x, w, scale, res) is None
        return
    want = (ops.linear_fp8(x, w, scale) if fp8 else ops.linear(x, w)) + res
    assert torch.equal(ops.linear_add(x, w, scale, res), want)
    if fp8:
        xq, xs = ops._require_ext("t").quantize_fp8_tensor(x)
        assert torch.equal(ops.linear_add(xq, w, scale, res, x_scale=xs), want)
        assert ops.linear_add(xq, w, scale, res) is None
    assert ops.linear_add(x, w, scale, res[:, :8]) is None
