"""The layers of a decode step in one launch, against the launches apart and both against
float64; steps that are not to take it."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from parallax_amd import ops
from parallax_amd.models import get_model_class
from parallax_amd.models.config import ModelConfig
from parallax_amd.models.forward_meta import ForwardMeta
from parallax_amd.server.kv_cache import KVCacheSpec, PagedKVCache


def _model(H, Hq, Hk, D, F, layers, bias=True, seed=0):
    cfg = ModelConfig(
        architecture="Qwen2ForCausalLM" if bias else "LlamaForCausalLM", vocab_size=64,
        hidden_size=H, num_layers=layers + 1, num_heads=Hq, num_kv_heads=Hk, head_dim=D,
        intermediate_size=F, max_position_embeddings=10240, attention_bias=bias,
        eos_token_ids=[])
    model = get_model_class(cfg.architecture)(cfg, 0, layers).to(torch.bfloat16).cuda()
    g = torch.Generator(device="cuda").manual_seed(seed)
    for name, p in model.named_parameters():
        scale = 0.1 if p.dim() == 1 else p.shape[1] ** -0.5 / (2 if "down" in name else 1)
        p.data.copy_(torch.randn(p.shape, generator=g, device="cuda") * scale)
        if "norm" in name:
            p.data += 1
    model.rope_cache = model.rope_cache.float().cuda()
    return model.eval(), cfg


def _step(cfg, layers, BS, lens, max_len=None, seed=1):
    """A step's input, its metadata on a cache of its own, and the cache."""
    assert max(lens) <= cfg.max_position_embeddings  # the kernels read the rope table there
    g = torch.Generator(device="cuda").manual_seed(seed)
    counts = [(max(n, 1) + BS - 1) // BS for n in lens]
    ids = torch.randperm(sum(counts), generator=g, device="cuda").tolist()
    bt = torch.zeros(len(lens), max(counts), dtype=torch.int32)
    at = 0
    for i, c in enumerate(counts):
        bt[i, :c] = torch.tensor(ids[at:at + c], dtype=torch.int32)
        at += c
    cache = PagedKVCache(KVCacheSpec(layers, cfg.num_kv_heads, cfg.head_dim, BS),
                         sum(counts), torch.device("cuda"))
    for t in cache.k_caches + cache.v_caches:
        t.copy_(torch.randn(t.shape, generator=g, device="cuda"))
    slots = [int(bt[i, (n - 1) // BS]) * BS + (n - 1) % BS if n else -1
             for i, n in enumerate(lens)]
    meta = ForwardMeta(
        is_prefill=False,
        positions=torch.tensor([max(n - 1, 0) for n in lens], dtype=torch.int32).cuda(),
        slot_mapping=torch.tensor(slots).cuda(), block_tables=bt.cuda(),
        seq_lens=torch.tensor(lens, dtype=torch.int32).cuda(), kv_cache=cache,
        max_seq_len=max_len or max(lens), appends=True)
    x = torch.randn(len(lens), cfg.hidden_size, generator=g, device="cuda").bfloat16()
    return x, meta, cache


@torch.inference_mode()
def _both(model, x, meta, cache, monkeypatch):
    """(result, K and V caches) in one launch and apart, from the same caches."""
    before = [t.clone() for t in cache.k_caches + cache.v_caches]
    calls, real = [], ops.decode_stack
    out = []
    for one in (True, False):
        for t, b in zip(cache.k_caches + cache.v_caches, before):
            t.copy_(b)
        with monkeypatch.context() as m:
            m.setattr(ops, "decode_stack", lambda *a: calls.append(real(*a)) or (
                calls[-1] if one else None))
            got = model(x.clone(), meta)
        assert (calls[-1] is not None) if one else True
        out.append((got.clone(), [t.clone() for t in cache.k_caches + cache.v_caches]))
    for t, b in zip(cache.k_caches + cache.v_caches, before):
        t.copy_(b)
    return out


def _exact(model, cfg, x, meta, cache, BS):
    """The step in float64 with the rounded values of weights and caches: the result, and
    each layer's rotated keys and values [M, Hk, D]."""
    h, D, Hq, Hk = x.double(), cfg.head_dim, cfg.num_heads, cfg.num_kv_heads

    def norm(v, w):
        return v * (v.pow(2).mean(-1, keepdim=True) + cfg.rms_norm_eps).rsqrt() * w.double()

    cs = model.rope_cache[meta.positions.long()].double()
    c, s = cs[:, None, :D // 2], cs[:, None, D // 2:]

    def turn(v):
        a, b = v[..., :D // 2], v[..., D // 2:]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    keys, values = [], []
    for i, layer in enumerate(model.layers):
        a = layer.self_attn
        qkv = norm(h, layer.input_layernorm.weight) @ a.qkv_proj.weight.double().T
        if a.qkv_proj.bias is not None:
            qkv = qkv + a.qkv_proj.bias.double()
        q, k, v = qkv.split([Hq * D, Hk * D, Hk * D], -1)
        q, k, v = turn(q.view(-1, Hq, D)), turn(k.view(-1, Hk, D)), v.view(-1, Hk, D)
        keys.append(k)
        values.append(v)
        rows = []
        for m, n in enumerate(meta.seq_lens.tolist()):
            if n == 0:
                rows.append(torch.zeros(Hq * D, dtype=torch.float64, device="cuda"))
                continue
            pages = meta.block_tables[m, :(n + BS - 1) // BS].long()
            kk = cache.k_caches[i][pages].transpose(1, 2).flatten(0, 1)[:n].double()
            vv = cache.v_caches[i][pages].permute(0, 3, 1, 2).flatten(0, 1)[:n].double()
            if meta.slot_mapping[m] >= 0:
                kk[-1], vv[-1] = k[m], v[m]
            kk, vv = (t.repeat_interleave(Hq // Hk, 1) for t in (kk, vv))
            p = (torch.einsum("hd,nhd->hn", q[m], kk) * a.scale).softmax(-1)
            rows.append(torch.einsum("hn,nhd->hd", p, vv).flatten())
        h = h + torch.stack(rows) @ a.o_proj.weight.double().T
        gu = norm(h, layer.post_attention_layernorm.weight) @ \
            layer.mlp.gate_up_proj.weight.double().T
        g, u = gu.chunk(2, -1)
        h = h + (torch.nn.functional.silu(g) * u) @ layer.mlp.down_proj.weight.double().T
    return h, keys, values


def _check_stored(kv, before, meta, keys, values, BS):
    """The step's tokens at their slots, with the keys and values of float64, and nothing
    else: all other places keep their bits.

    The first layer's are off by what the norm, the product and the rotation round, each
    by at most 2^-9 of a value: 2^-7 of their norm is above all three. A layer further on
    adds as much to the stream, independently: the squares add up."""
    n = len(kv) // 2
    rows = (meta.slot_mapping >= 0).nonzero()[:, 0]
    slots = meta.slot_mapping[rows]
    page, at = slots // BS, slots % BS
    for i in range(n):
        for got, old, want, tokens in ((kv[i], before[i], keys[i], 2),
                                       (kv[n + i], before[n + i], values[i], 3)):
            got, old = (t.movedim(tokens, 1) for t in (got, old))  # [page, token, Hk, D]
            rest = torch.ones(got.shape[:2], dtype=torch.bool, device="cuda")
            rest[page, at] = False
            assert torch.equal(got[rest].view(torch.int16), old[rest].view(torch.int16))
            want = want[rows]
            err = (got[page, at].double() - want).norm(dim=(1, 2))
            assert (err <= 2 ** -7 * (i + 1) ** 0.5 * want.norm(dim=(1, 2))).all(), i


CASES = [
    # H, Hq, Hk, D, F, layers, BS, lengths
    (896, 14, 2, 64, 4864, 2, 32, [600]),
    (32, 1, 1, 64, 32, 3, 16, [1]),                      # one step along K, one tile
    (64, 15, 1, 64, 96, 2, 64, [31, 257]),               # all columns but one are heads
    (1024, 8, 8, 128, 5120, 1, 32, [33, 1024, 1]),       # the widest
    (992, 16, 4, 64, 4000, 2, 16, [255, 256, 2500, 17]),  # steps that leave waves short
    (160, 6, 2, 128, 1056, 2, 64, [4096, 2]),
    (288, 3, 3, 64, 480, 35, 32, [70, 300]),             # a second launch
    (96, 4, 2, 64, 224, 2, 32, [0, 5, 0]),               # rows without tokens
]


@pytest.mark.parametrize("H,Hq,Hk,D,F,layers,BS,lens", CASES)
def test_decode_stack(H, Hq, Hk, D, F, layers, BS, lens, monkeypatch):
    """Against float64 no further off than the launches apart: the same roundings, of sums
    in another order. Single roundings fall either way; 1.25 of the norm of many values,
    with few of them more: a norm of n independent errors is known to 1 / sqrt(2 n)."""
    model, cfg = _model(H, Hq, Hk, D, F, layers, bias=layers % 2 == 0)
    x, meta, cache = _step(cfg, layers, BS, lens)
    want, keys, values = _exact(model, cfg, x, meta, cache, BS)
    (one, kv1), (apart, kv2) = _both(model, x, meta, cache, monkeypatch)
    e1, e2 = ((t.double() - want).norm() for t in (one, apart))
    assert e1 <= e2 * (1.25 + 4 / (2 * want.numel()) ** 0.5)
    before = _step(cfg, layers, BS, lens)[2]
    for kv in (kv1, kv2):
        _check_stored(kv, before.k_caches + before.v_caches, meta, keys, values, BS)


def test_decode_stack_over_stale_slots(monkeypatch):
    """The token's own place and those behind it hold NaN; one row's token is cached."""
    model, cfg = _model(256, 4, 2, 64, 512, 2)
    lens = [40, 33, 300]
    x, meta, cache = _step(cfg, 2, 32, lens)
    for m, n in enumerate(lens):
        page, at = int(meta.block_tables[m, (n - 1) // 32]), (n - 1) % 32
        if m == 1:
            meta.slot_mapping[1], at = -1, at + 1
        for k, v in zip(cache.k_caches, cache.v_caches):
            k[page, :, at:] = float("nan")
            v[page, :, :, at:] = float("nan")
    want, keys, values = _exact(model, cfg, x, meta, cache, 32)
    before = [t.clone() for t in cache.k_caches + cache.v_caches]
    (one, kv), (apart, _) = _both(model, x, meta, cache, monkeypatch)
    _check_stored(kv, before, meta, keys, values, 32)
    assert one.isfinite().all()
    assert (one.double() - want).norm() <= 1.4 * (apart.double() - want).norm()


def test_decode_stack_infinities(monkeypatch):
    """Infinite weights reach the results they belong to and no others."""
    model, cfg = _model(992, 4, 2, 64, 480, 1)
    x, meta, cache = _step(cfg, 1, 32, [50, 20])
    w = model.layers[0].mlp.down_proj.weight
    w.data[7, 479] = float("inf")
    w.data[20, 0] = float("-inf")
    (one, _), (apart, _) = _both(model, x, meta, cache, monkeypatch)
    assert torch.equal(one.isfinite(), apart.isfinite())
    assert not one[:, [7, 20]].isfinite().any()
    assert one[:, [i for i in range(992) if i not in (7, 20)]].isfinite().all()


@torch.inference_mode()
def test_decode_stack_in_a_graph():
    """Each replay takes the lengths, places and values of then; eager steps between them
    on the same and on another stream change nothing."""
    model, cfg = _model(896, 14, 2, 64, 1024, 4)
    x, meta, cache = _step(cfg, 4, 32, [700, 40], max_len=1024)
    model(x, meta)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = model(x, meta)
    side = torch.cuda.Stream()
    for step in range(4):
        meta.seq_lens.sub_(3)
        meta.positions.sub_(3)
        n = meta.seq_lens - 1
        meta.slot_mapping.copy_(
            meta.block_tables.gather(1, (n // 32).long()[:, None])[:, 0] * 32 + n % 32)
        x.mul_(-0.75)
        want = model(x, meta).clone()
        kv = [t.clone() for t in cache.k_caches + cache.v_caches]
        torch.cuda.synchronize()
        with torch.cuda.stream(side):  # both at once: each has its own words
            graph.replay()
        again = model(x, meta)
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(again, want)
        assert all(torch.equal(a, b) for a, b in zip(kv, cache.k_caches + cache.v_caches))


@pytest.mark.parametrize("M,D,last", [
    (1, 64, 16384), (2, 64, 8192), (3, 64, 4096), (4, 64, 4096),
    (1, 128, 8192), (2, 128, 4096), (3, 128, 2048), (4, 128, 2048),
])
def test_contexts_up_to_what_a_workgroup_takes_in_turn(M, D, last):
    """Eight units of 256 tokens a part of 64-wide heads, four of 128-wide ones."""
    for n, has in ((1, True), (last, True), (last + 1, False)):
        assert ops.decode_stack_has(M, 896, 512 // D, 2, D, 4864, n) == has


def test_decode_stack_is_left(monkeypatch):
    """What is more than plain layers, or beyond the kernel's sizes, goes the other way."""
    took = []
    real = ops.decode_stack
    monkeypatch.setattr(ops, "decode_stack",
                        lambda *a: took.append(real(*a)) or took[-1])

    def run(change=None, lens=(40, 9), sizes=(256, 4, 2, 64, 512), **kw):
        model, cfg = _model(*sizes, 2)
        x, meta, _ = _step(cfg, 2, 32, list(lens))
        for k, v in kw.items():
            setattr(meta, k, v)
        if change:
            change(model)
        took.clear()
        with torch.inference_mode():
            model(x, meta)
        return bool(took) and took[-1] is not None

    assert run()
    assert not run(appends=False)
    assert not run(lens=[5] * 5)
    assert not run(lens=[20, 8500])
    assert not run(sizes=(1056, 4, 2, 64, 512))
    assert not run(sizes=(256, 4, 2, 64, 5152))
    seen = []
    assert not run(lambda m: m.layers[1].mlp.register_forward_hook(
        lambda *a: seen.append(1)))
    assert seen
    assert not run(lambda m: m.layers[1].self_attn.o_proj.quantize_fp8())
    assert not run(lambda m: setattr(m.layers[1].self_attn, "sliding_window", 16))
    assert not run(lambda m: setattr(m.layers[1].post_attention_layernorm, "eps", 1e-3))


class _Norm(torch.nn.Module):
    """A norm of a caller's own: no RMSNorm, no eps."""

    def __init__(self, norm):
        super().__init__()
        self.inner = norm

    def forward(self, x, residual=None):
        return self.inner(x, residual)


@pytest.mark.parametrize("layer", [0, 1])
@pytest.mark.parametrize("name", ["input_layernorm", "post_attention_layernorm"])
def test_other_norms_run(layer, name):
    """A step over modules that stand in a norm's place, as the layers themselves take
    them, gives what it gives over the norms apart."""
    model, cfg = _model(256, 4, 2, 64, 512, 2)
    x, meta, _ = _step(cfg, 2, 32, [40, 9])
    seen = []
    with torch.inference_mode():
        hooked = getattr(model.layers[layer], name)
        handle = hooked.register_forward_hook(lambda *a: seen.append(1))
        want = model(x.clone(), meta).clone()
        handle.remove()
        assert seen
        setattr(model.layers[layer], name, _Norm(hooked))
        assert torch.equal(model(x.clone(), meta), want)


def test_a_row_of_three_dimensions_runs():
    """[1, 1, H] goes through the layers, whose results are bf16: 2^-6 of their norm is
    four roundings of a value a layer."""
    model, cfg = _model(256, 4, 2, 64, 512, 2)
    x, meta, _ = _step(cfg, 2, 32, [40])
    with torch.inference_mode():
        want = model(x.clone(), meta).float()
        got = model(x[None].clone(), meta)
    assert got.shape == (1, 1, 256)
    assert (got[0].float() - want).norm() <= 2 ** -6 * want.norm()


def test_a_step_refused_as_a_whole_is_refused_early(monkeypatch):
    """fp8 caches, rope of part of a head and a gradient to be taken are seen before the
    layers are: the host pays for none of them."""
    model, cfg = _model(256, 4, 2, 64, 512, 2)
    monkeypatch.setattr(ops, "decode_stack", lambda *a: pytest.fail("asked"))
    x, meta, cache = _step(cfg, 2, 32, [40, 9])
    with torch.enable_grad():
        model(x.clone().requires_grad_(), meta)
    with torch.inference_mode():
        with monkeypatch.context() as m:
            m.setattr(model, "rope_cache", model.rope_cache[:, :32].contiguous())
            model(x.clone(), meta)
        meta.kv_cache = PagedKVCache(KVCacheSpec(2, 2, 64, 32, torch.float8_e4m3fn),
                                     len(cache.k_caches[0]), torch.device("cuda"))
        model(x.clone(), meta)
        meta.kv_cache = cache
        with pytest.raises(pytest.fail.Exception):
            model(x.clone(), meta)
