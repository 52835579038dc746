"""Norm and product of a few rows in one launch, against float64 and against the two
launches; a layer that takes it against the same layer with hooks, which does not."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from parallax_amd import ops


def _rand(g, *s):
    return torch.randn(*s, generator=g, device="cuda").bfloat16()


@pytest.mark.parametrize("M,N,K", [
    (M, N, K) for M in (1, 3, 4) for N, K in (
        (1, 32), (17, 512),            # less than a tile; waves without a step
        (1152, 896), (2050, 928), (18000, 1024),   # four waves; tiles in turn
        (100, 1056), (512, 1536), (9000, 1568), (36, 2048),  # eight
    )
] + [(1, 48, 2080), (2, 5000, 3072), (2, 70, 3104), (1, 4100, 4096)])
def test_norm_linear(M, N, K):
    """The normed rows are rounded to bf16 from fp32 values a few 2^-24 off: a value
    may round to its neighbour, 2^-8 of it, against float64. So each result is within
    its own rounding, 2^-9, and 2^-8 of the norm of the terms (sum (h w)^2)^1/2 a few
    times; gated products of two such a few times more."""
    g = torch.Generator(device="cuda").manual_seed(M * N + K)
    x, res = _rand(g, M, K + 8)[:, 8:], _rand(g, M, K) * 3
    norm, w, b = 1 + 0.1 * _rand(g, K), _rand(g, N, K) * K ** -0.5, _rand(g, N)
    for residual in (res, None):
        for bias in (b, None):
            got = ops.norm_linear(x, residual, norm, 1e-5, w, bias)
            s = x if residual is None else (x.float() + residual.float()).bfloat16()
            assert torch.equal(got[1], s)
            raw = x.double() if residual is None else x.double() + residual.double()
            h = s.double() * (raw.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt()
            h = (h * norm.double()).bfloat16().double()
            want = h @ w.double().T + (0 if bias is None else bias.double())
            terms = (h.pow(2) @ w.double().pow(2).T).sqrt()
            assert ((got[0].double() - want).abs()
                    <= 2 ** -8 * want.abs() + 2 ** -6 * terms).all()
    if N % 2 == 0:
        a, u = want[:, :N // 2], want[:, N // 2:]   # without a bias
        got = ops.norm_linear(x, None, norm, 1e-5, w, None, gated=True)[0]
        silu = torch.nn.functional.silu(a)
        terms = terms[:, :N // 2] * (u.abs() + 1) + terms[:, N // 2:] * (a.abs() + 1)
        assert ((got.double() - silu * u).abs()
                <= 2 ** -6 * (silu * u).abs() + 2 ** -5 * terms).all()
    if K <= 1536:  # the product alone, through linear
        want = x.double() @ w.double().T + b.double()
        torch.testing.assert_close(ops.linear(x, w, b).double(), want, rtol=2 ** -8,
                                   atol=K * 2 ** -20)


@pytest.mark.parametrize("K", [32, 480, 928, 1056, 1568, 2048, 2080, 3104, 3584])
def test_norm_linear_infinities(K):
    """An infinite weight of the last column or the first makes its row's results
    infinite, with the sign of the value it meets, and no other's; also where the steps
    along K leave waves of the last ones without any."""
    g = torch.Generator(device="cuda").manual_seed(K)
    x, norm, w = _rand(g, 2, K), torch.ones(K, device="cuda").bfloat16(), _rand(g, 70, K)
    x[:, 0] = x[:, -1] = torch.tensor([1.0, -1.0])
    for row, col in ((3, -1), (17, 0), (69, -1)):
        w[row, col] = float("inf")
    outs = [ops.norm_linear(x, None, norm, 1e-5, w)[0],
            ops.norm_linear(x, x, norm, 1e-5, w)[0]]
    if K <= 1536:
        outs.append(ops.linear(x, w))
    for out in outs:
        for row in (3, 17, 69):
            assert out[:, row].tolist() == [float("inf"), float("-inf")]
        out[:, [3, 17, 69]] = 0
        assert out.isfinite().all()


def test_norm_linear_without_a_kernel():
    g = torch.Generator(device="cuda").manual_seed(0)
    x, w, n = _rand(g, 2, 64), _rand(g, 32, 64), _rand(g, 64)
    assert ops.norm_linear(x, None, n, 1e-5, w) is not None
    assert ops.norm_linear(_rand(g, 5, 64), None, n, 1e-5, w) is None
    assert ops.norm_linear(_rand(g, 2, 68)[:, 4:], None, n, 1e-5, w) is None
    assert ops.norm_linear(x, None, n, 1e-5, w.float()) is None
    assert ops.norm_linear(x, _rand(g, 1, 64), n, 1e-5, w) is None
    assert ops.norm_linear(x, None, n, 1e-5, w, _rand(g, 1)) is None
    assert ops.norm_linear(x[:0], None, n, 1e-5, w) is None
    assert ops.norm_linear(x, None, n, 1e-5, w.requires_grad_()) is None


@pytest.mark.parametrize("T", [1, 4, 5])
def test_gated_parts_of_odd_widths_are_refused(T):
    """Of any number of rows alike: silu_and_mul takes parts of multiples of 8."""
    from parallax_amd.models.llama import RMSNorm, norm_project
    from parallax_amd.parallel.layers import MergedColumnParallelLinear
    g = torch.Generator(device="cuda").manual_seed(0)
    x, w = _rand(g, T, 64), _rand(g, 24, 64)
    with pytest.raises(RuntimeError):
        ops.linear_silu_and_mul(x, w)
    with torch.device("cuda"):
        norm = RMSNorm(64, 1e-5).bfloat16()
        proj = MergedColumnParallelLinear(64, [12, 12]).bfloat16()
        wide = MergedColumnParallelLinear(64, [16, 16]).bfloat16()
    with torch.no_grad():
        assert norm_project(norm, proj, x, None, gated=True) is None
        assert (norm_project(norm, proj, x, None) is None) == (T > 4)
        assert (norm_project(norm, wide, x, None, gated=True) is None) == (T > 4)


def _shard(**kw):
    from parallax_amd.models import get_model_class
    from parallax_amd.models.config import ModelConfig
    cfg = ModelConfig(**{**dict(
        architecture="Qwen2ForCausalLM", vocab_size=128, hidden_size=256, num_layers=2,
        num_heads=4, num_kv_heads=2, head_dim=64, intermediate_size=320,
        max_position_embeddings=256, attention_bias=True, eos_token_ids=[]), **kw})
    with torch.device("cuda"):
        model = get_model_class(cfg.architecture)(cfg, 0, 2).to(torch.bfloat16)
    model.rope_cache = model.rope_cache.float().cuda()
    torch.manual_seed(0)
    for name, p in model.named_parameters():
        p.data.copy_(torch.randn(p.shape) * (0.1 if p.dim() > 1 else 0.3)
                     + (1 if "norm" in name else 0))
    return cfg, model


def _step(cfg, model, T):
    from parallax_amd.models.forward_meta import ForwardMeta
    from parallax_amd.server.kv_cache import KVCacheSpec, PagedKVCache
    dev = torch.device("cuda")
    cache = PagedKVCache(KVCacheSpec(2, 2, 64, 16), 8, dev)
    g = torch.Generator(device="cuda").manual_seed(T)
    for c in cache.k_caches + cache.v_caches:
        c.copy_(torch.randn(c.shape, generator=g, device="cuda"))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    meta = ForwardMeta(
        is_prefill=False, positions=i32([5 + i for i in range(T)]),
        slot_mapping=torch.tensor([16 * i + 5 + i for i in range(T)], device=dev),
        block_tables=i32([[i] for i in range(T)]),
        seq_lens=i32([6 + i for i in range(T)]), query_lens=None, kv_cache=cache,
        logits_indices=None, max_seq_len=16)
    ids = torch.arange(T, device=dev) * 7
    with torch.inference_mode():
        return model(model.embed(ids), meta), cache


@pytest.mark.parametrize("T", [1, 4, 5])
@pytest.mark.parametrize("where", ["input_layernorm", "self_attn.qkv_proj", "self_attn",
                                   "post_attention_layernorm", "mlp.gate_up_proj",
                                   "mlp"])
def test_a_hook_sees_what_it_would(T, where):
    """The hooked module runs on the normed rows; the step's results differ by
    roundings of bf16 values on the way only (2^-8 each, some ten of them)."""
    cfg, model = _shard()
    want, cache = _step(cfg, model, T)
    seen = []
    model.layers[1].get_submodule(where).register_forward_hook(
        lambda m, args, out: seen.append(args[0].shape))
    got, cache2 = _step(cfg, model, T)
    assert seen == [(T, 256)]
    assert (got - want).norm() < 2 ** -5 * want.norm()
    for a, b in zip(cache.k_caches + cache.v_caches, cache2.k_caches + cache2.v_caches):
        assert (a.float() - b.float()).norm() < 2 ** -5 * b.float().norm()
