"""MLA decode kernel numerics vs fp32 reference + DeepSeek GPU engine smoke."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from parallax_amd import ops
from parallax_amd.ops import reference as ref


def _setup(B, H, ctxs, R=512, DR=64, BS=32, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    max_blocks = (max(ctxs) + BS - 1) // BS
    NB = B * max_blocks + 1
    cache = torch.randn(NB, BS, R + DR, generator=g, dtype=torch.bfloat16,
                        device="cuda")
    bt = (
        torch.arange(B * max_blocks, dtype=torch.int32, device="cuda")
        .reshape(B, max_blocks) + 1
    )
    ql = torch.randn(B, H, R, generator=g, dtype=torch.bfloat16, device="cuda") * 0.1
    qp = torch.randn(B, H, DR, generator=g, dtype=torch.bfloat16, device="cuda") * 0.1
    sl = torch.tensor(ctxs, dtype=torch.int32, device="cuda")
    return ql, qp, cache, bt, sl


@pytest.mark.parametrize("H,ctxs", [
    (128, [100, 37]),          # deepseek-v3 head count, short ctx
    (128, [1025, 300]),        # partitioned path
    (32, [64]),                # single head block
    (16, [1, 500]),            # H < HBLOCK (padded columns)
])
def test_mla_decode_kernel(H, ctxs):
    ql, qp, cache, bt, sl = _setup(len(ctxs), H, ctxs)
    scale = 1.0 / math.sqrt(128 + 64)
    out = ops.mla_paged_attention_decode(ql, qp, cache, bt, sl, scale)
    expect = ref.mla_paged_attention_decode(
        ql.float().cpu(), qp.float().cpu(), cache.float().cpu(), bt.cpu(),
        sl.cpu(), scale,
    )
    torch.testing.assert_close(
        out.float().cpu(), expect.float().cpu(), atol=6e-2, rtol=6e-2
    )


def test_deepseek_engine_gpu_smoke():
    """Tiny DeepSeek-shaped model (kv_lora 512/rope 64 geometry) decodes on the
    HIP MLA kernel end-to-end."""
    from parallax_amd.models.config import ModelConfig
    from parallax_amd.server.engine import Engine, EngineArgs
    from parallax_amd.server.sampling_params import SamplingParams

    cfg = ModelConfig(
        architecture="DeepseekV3ForCausalLM", model_type="deepseek_v3",
        vocab_size=512, hidden_size=256, num_layers=2, num_heads=16,
        num_kv_heads=16, head_dim=64, intermediate_size=512,
        moe_intermediate_size=128, num_experts=4, num_experts_per_tok=2,
        num_shared_experts=1, first_k_dense_layers=1, scoring_func="sigmoid",
        n_group=0, topk_group=0,
        q_lora_rank=128, kv_lora_rank=512, qk_nope_head_dim=64,
        qk_rope_head_dim=64, v_head_dim=64,
        max_position_embeddings=2048, eos_token_ids=[],
    )
    eng = Engine(cfg, EngineArgs(num_kv_blocks=128), random_weights=True)
    out = eng.generate(
        [[1, 2, 3, 4, 5, 6, 7, 8], [9] * 40],
        [SamplingParams(temperature=0.0, max_new_tokens=5, ignore_eos=True)] * 2,
    )
    assert all(len(v) == 5 for v in out.values())


@pytest.mark.gpu
def test_mla_decode_fp8_cache():
    """FP8-E4M3 compressed cache: quantize-on-store + dequantize-in-staging
    must track the bf16 kernel within fp8 rounding error."""
    torch.manual_seed(3)
    B, H, R, DR, BS = 4, 32, 512, 64, 32
    ctxs = [300, 77, 512, 40]
    max_blocks = (max(ctxs) + BS - 1) // BS
    NB = B * max_blocks + 1
    latent = torch.randn(sum(ctxs), R, dtype=torch.bfloat16, device="cuda") / 4
    rope = torch.randn(sum(ctxs), DR, dtype=torch.bfloat16, device="cuda") / 4
    cache8 = torch.zeros(NB, BS, R + DR, dtype=torch.float8_e4m3fn, device="cuda")
    cache16 = torch.zeros(NB, BS, R + DR, dtype=torch.bfloat16, device="cuda")
    bt = (torch.arange(B * max_blocks, dtype=torch.int32, device="cuda")
          .reshape(B, max_blocks) + 1)
    slots = []
    t0 = 0
    for i, L in enumerate(ctxs):
        for p in range(L):
            blk = int(bt[i, p // BS])
            slots.append(blk * BS + p % BS)
        t0 += L
    sm = torch.tensor(slots, dtype=torch.int64, device="cuda")
    ops.mla_reshape_and_cache(latent, rope, cache8, sm)
    ops.mla_reshape_and_cache(latent, rope, cache16, sm)
    sl = torch.tensor(ctxs, dtype=torch.int32, device="cuda")
    ql = torch.randn(B, H, R, dtype=torch.bfloat16, device="cuda") / 8
    qp = torch.randn(B, H, DR, dtype=torch.bfloat16, device="cuda") / 8
    scale = 1.0 / math.sqrt(R + DR)
    out8 = ops.mla_paged_attention_decode(ql, qp, cache8, bt, sl, scale)
    out16 = ops.mla_paged_attention_decode(ql, qp, cache16, bt, sl, scale)
    # fp8 rounding on both K and V sides: loose tolerance, but the softmax
    # keeps outputs in the same range
    torch.testing.assert_close(out8.float(), out16.float(), atol=0.12, rtol=0.12)
    # and the fp8 store actually quantized (bytes differ from bf16 view)
    assert cache8.dtype == torch.float8_e4m3fn


@pytest.mark.parametrize("H,BS,ctxs,fp8", [
    (16, 16, [1, 31, 33, 700], False),     # runs that cross sequences
    (40, 32, [5000, 64, 3], False),        # one sequence over many runs
    (128, 64, [600, 90, 1500], False),
    (200, 32, [300, 257], False),          # more heads than a workgroup takes
    (24, 32, [250] * 3, False),            # a workgroup a sequence
    (64, 16, [47, 900], True),
    (128, 32, [333, 70], True),
])
def test_mla_decode_runs(H, BS, ctxs, fp8):
    """Tiles dealt over sequences, every page size and head count per wave,
    cache slots behind a sequence's end holding NaN. Weights and results are
    rounded to bf16 once each: at most 2 * 2^-9 * max |cache| (5.5)."""
    ql, qp, cache, bt, sl = _setup(len(ctxs), H, ctxs, BS=BS, seed=H)
    ql, qp = ql * 10, qp * 10
    if fp8:
        cache = cache.to(torch.float8_e4m3fn)
    plain = cache.float()
    for i, n in enumerate(ctxs):
        if n % BS and not fp8:
            cache[int(bt[i, n // BS]), n % BS:] = float("nan")
    scale = 192 ** -0.5
    out = ops.mla_paged_attention_decode(ql, qp, cache, bt, sl, scale)
    want = ref.mla_paged_attention_decode(
        ql.float().cpu(), qp.float().cpu(), plain.cpu(), bt.cpu(), sl.cpu(), scale)
    torch.testing.assert_close(out.float().cpu(), want, atol=2.2e-2, rtol=0)


@pytest.mark.parametrize("H", [16, 72, 128])
@pytest.mark.parametrize("max_seq_len", [200, 4096, 10 ** 6])
def test_mla_decode_sequences_without_tokens(H, max_seq_len):
    """Results of 0, whatever the memory held; the others as ever."""
    ctxs = [0, 130, 0, 0, 7, 0] * (4 if max_seq_len == 10 ** 6 else 1)
    ql, qp, cache, bt, sl = _setup(len(ctxs), H, ctxs, seed=H)
    poison = [torch.full_like(ql, float("nan")) for _ in range(8)]
    del poison
    scale = 192 ** -0.5
    out = ops.mla_paged_attention_decode(ql, qp, cache, bt, sl, scale,
                                         max_seq_len=max_seq_len)
    want = torch.zeros(ql.shape)
    some = [i for i, n in enumerate(ctxs) if n]
    want[some] = ref.mla_paged_attention_decode(
        ql[some].float().cpu(), qp[some].float().cpu(), cache.float().cpu(),
        bt[some].cpu(), sl[some].cpu(), scale)
    torch.testing.assert_close(out.float().cpu(), want, atol=2.2e-2, rtol=0)


@pytest.mark.parametrize("H,topk", [(16, 40), (128, 512)])
def test_mla_decode_listed_tokens(H, topk):
    """Rows restricted to listed positions (some entries stand for none), beside
    a row without a list."""
    ctxs = [700, 90, 1300]
    ql, qp, cache, bt, sl = _setup(3, H, ctxs, seed=topk)
    ql = ql * 10
    idx = torch.full((3, topk), -1, dtype=torch.int32)
    g = torch.Generator().manual_seed(1)
    for i, n in enumerate(ctxs):
        k = min(topk, n) - 7
        idx[i, :k] = torch.randperm(n, generator=g)[:k].int()
    idx[0, 11] = -1
    idx[1, 0] = -1                          # attends to everything
    scale = 192 ** -0.5
    out = ops.dsa_paged_attention_decode(ql, qp, cache, bt, sl, idx.cuda(), scale)
    want = ref.dsa_paged_attention_decode(
        ql.float().cpu(), qp.float().cpu(), cache.float().cpu(), bt.cpu(),
        sl.cpu(), idx, scale)
    torch.testing.assert_close(out.float().cpu(), want, atol=2.2e-2, rtol=0)


@pytest.mark.parametrize("fp8", [False, True])
def test_mla_decode_list_without_tokens(fp8):
    """A list beside an empty sequence, whose table row holds a page that is not
    there: no page is read for it, its result is 0."""
    ql, qp, cache, bt, sl = _setup(3, 16, [300, 300, 300], seed=3)
    ql, idx = ql * 10, torch.full((3, 70), -1, dtype=torch.int32, device="cuda")
    idx[:, :40] = torch.arange(0, 280, 7, dtype=torch.int32, device="cuda")
    if fp8:
        cache = cache.to(torch.float8_e4m3fn)
    bt[1], sl[1] = -1, 0
    out = ops.dsa_paged_attention_decode(ql, qp, cache, bt, sl, idx, 192 ** -0.5)
    assert float(out[1].abs().max()) == 0
    want = ref.dsa_paged_attention_decode(
        ql[::2].float(), qp[::2].float(), cache.float(), bt[::2], sl[::2], idx[::2],
        192 ** -0.5)
    torch.testing.assert_close(out[::2].float(), want, atol=2.2e-2, rtol=0)


@pytest.mark.parametrize("H,T,L,fp8", [
    (128, 1, 1, False),
    (8, 33, 33, False),           # past a wave's 32 rows and a tile's 32 keys
    (16, 127, 160, True),
    (16, 129, 1000, False),       # past a workgroup's 128 rows
    (128, 130, 8192 + 40, False), # a second run of expanded rows, the
                                  # portion's first rows before it
])
def test_mla_prefill(H, T, L, fp8):
    """Against fp32 products. The result's rounding is 2^-8 of it at most; a logit is
    off by at most the lo parts' rounding, sum |q k| * scale * 2^-17 < 2e-4,
    a result by twice that of max |v| < 6."""
    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    q = r(T, H, 192).bfloat16()
    q_nope, q_pe = q[..., :128], q[..., 128:].contiguous()
    rows = r(L, 576).to(torch.float8_e4m3fn if fp8 else torch.bfloat16)
    uk, uv = ((r(H, 128, 512) * 512 ** -0.5).bfloat16() for _ in range(2))
    out = torch.empty(T, H, 128, dtype=torch.bfloat16, device="cuda")
    scale = 192 ** -0.5
    assert ops.mla_prefill_attention(out, q_nope, q_pe, rows, uk, uv, scale)
    e = rows.float()
    hidden = torch.arange(L, device="cuda")[None] > torch.arange(
        L - T, L, device="cuda")[:, None]
    for h in {0, H // 2, H - 1}:
        k, v = e[:, :512] @ uk[h].float().t(), e[:, :512] @ uv[h].float().t()
        s = q_nope[:, h].float() @ k.t() + q_pe[:, h].float() @ e[:, 512:].t()
        p = (s * scale).masked_fill(hidden, float("-inf")).softmax(-1)
        torch.testing.assert_close(
            out[:, h].float(), p @ v, atol=2.4e-3, rtol=2 ** -8)


@pytest.mark.parametrize("scale", [-0.07, 0.0])
def test_mla_prefill_scales_of_any_sign(scale):
    """Below 0 and 0 (a plain mean): hidden keys have no weight either way. 3 heads,
    130 rows on 170, tolerance as above."""
    g = torch.Generator(device="cuda").manual_seed(5)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    H, T, L = 3, 130, 300
    q_nope, q_pe = r(T, H, 128).bfloat16(), r(T, H, 64).bfloat16()
    rows = r(L, 576).bfloat16()
    uk, uv = ((r(H, 128, 512) * 512 ** -0.5).bfloat16() for _ in range(2))
    out = torch.empty(T, H, 128, dtype=torch.bfloat16, device="cuda")
    assert ops.mla_prefill_attention(out, q_nope, q_pe, rows, uk, uv, scale)
    e = rows.float()
    hidden = torch.arange(L, device="cuda")[None] > torch.arange(
        L - T, L, device="cuda")[:, None]
    for h in range(H):
        k, v = e[:, :512] @ uk[h].float().t(), e[:, :512] @ uv[h].float().t()
        s = q_nope[:, h].float() @ k.t() + q_pe[:, h].float() @ e[:, 512:].t()
        p = (s * scale).masked_fill(hidden, float("-inf")).softmax(-1)
        torch.testing.assert_close(
            out[:, h].float(), p @ v, atol=2.4e-3, rtol=2 ** -8)


@pytest.mark.parametrize("H,page,lens", [
    (128, 64, [(1, 1)]),
    (16, 16, [(33, 33), (0, 40), (129, 1000), (127, 127)]),  # out of order, one without rows
    (3, 32, [(130, 300), (256, 256), (1, 129)]),             # heads that XCDs do not share
    (16, 16, [(5 + 13 * i, 5 + 17 * i) for i in range(19)]), # more than a launch takes
    (128, 128, [(60, 5000), (300, 3500), (7, 20)]),          # more rows than it expands
])
def test_mla_prefill_of_all_requests(H, page, lens):
    """The bits of a request at a time, from shuffled pages whose unused slots hold NaN."""
    g = torch.Generator(device="cuda").manual_seed(H + len(lens))
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T = sum(n for n, _ in lens)
    q = r(T, H, 192).bfloat16()
    q_nope, q_pe = q[..., :128], q[..., 128:].contiguous()
    uk, uv = ((r(H, 128, 512) * 512 ** -0.5).bfloat16() for _ in range(2))
    counts = [-(-n // page) for _, n in lens]
    cache = torch.full((sum(counts) + 3, page, 576), float("nan"), device="cuda").bfloat16()
    ids = torch.randperm(sum(counts), generator=g, device="cuda").int()
    tables = torch.full((len(lens), max(counts) + 2), 1 << 30, dtype=torch.int32,
                        device="cuda")
    out = torch.empty(T, H, 128, dtype=torch.bfloat16, device="cuda")
    want, at, row = torch.empty_like(out), 0, 0
    for i, (n, context) in enumerate(lens):
        mine = ids[at:at + counts[i]]
        at += counts[i]
        tables[i, :counts[i]] = mine
        rows = r(context, 576).bfloat16()
        for j in range(counts[i]):
            part = rows[j * page:(j + 1) * page]
            cache[mine[j].item(), :len(part)] = part
        part = slice(row, row + n)
        row += n
        if n:
            assert ops.mla_prefill_attention(want[part], q_nope[part], q_pe[part], rows,
                                             uk, uv, 192 ** -0.5)
    assert ops.mla_prefill_paged(out, q_nope, q_pe, cache, tables, lens, uk, uv,
                                 192 ** -0.5)
    assert torch.equal(out, want)
    for lens, cache, tables in (
        (lens, cache.float(), tables), (lens, cache.to(torch.float8_e4m3fn), tables),
        (lens, cache[..., :512], tables), (lens, cache[:, :page - 1], tables),
        (lens, cache, tables.long()), (lens, cache, tables[:, :max(counts) - 1]),
        ([(lens[0][0], (1 << 20) // H + 128)] + lens[1:], cache, tables),  # by runs
        (lens + [(1, 1)], cache, tables),
    ):
        assert not ops.mla_prefill_paged(out, q_nope, q_pe, cache, tables, lens, uk, uv, 1.0)


def test_mla_prefill_left_to_the_caller():
    """Types, widths and few rows on a long context have no kernel."""
    def call(T, L, H=16, dtype=torch.bfloat16, dn=128, dr=64, dev="cuda"):
        z = lambda *s: torch.zeros(*s, dtype=dtype, device=dev)
        return ops.mla_prefill_attention(
            z(T, H, 128), z(T, H, dn), z(T, H, dr), z(L, 512 + dr),
            z(H, dn, 512), z(H, 128, 512), 1.0)
    assert call(40, 40)
    assert not call(4, 30000)
    assert not call(40, 40, dtype=torch.float32)
    assert not call(40, 40, dn=64)
    assert not call(40, 40, dr=32)
    assert not call(40, 40, dev="cpu")


def test_mla_prefill_operands_in_other_orders_left_to_the_caller():
    """Views of a fused weight, a result or a context that is not the kernel's."""
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")
    q, pe, rows, w = z(40, 16, 128), z(40, 16, 64), z(50, 576), z(16, 128, 512)
    fused = z(16, 256, 512)
    assert ops.mla_prefill_attention(z(40, 16, 128), q, pe, rows, w, w, 1.0)
    for out, r, uk, uv in (
        (z(40, 16, 128), rows, fused[:, :128], w),
        (z(40, 16, 128), rows, w, fused[:, 128:]),
        (z(40, 16, 256)[..., :128], rows, w, w),
        (z(40, 16, 128), rows[:39], w, w),      # a portion longer than its context
    ):
        assert not ops.mla_prefill_attention(out, q, pe, r, uk, uv, 1.0)


@pytest.mark.parametrize("T,H,R,DR", [(1, 128, 512, 64), (5, 3, 64, 16), (70, 16, 512, 64),
                                      (3, 33, 1032, 128)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("neox", [False, True])
def test_mla_rope_and_cache(T, H, R, DR, fp8, neox):
    """The same bits as its five steps: sums of squares run in the same order."""
    g = torch.Generator(device="cuda").manual_seed(T)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    q, kv, w = rand(T, H, DR + 32)[..., 32:], rand(T, R + DR + 8)[:, :R + DR], rand(R)
    table = torch.randn(90, DR, generator=g, device="cuda")
    pos = torch.randint(0, 90, (T,), generator=g, device="cuda", dtype=torch.int32)
    slots = torch.randperm(96, generator=g, device="cuda")[:T]
    slots[T // 2] = -1
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    caches = [torch.zeros(6, 16, R + DR, device="cuda").to(dt) for _ in range(2)]
    got = ops.mla_rope_and_cache(q, kv, w, 1e-6, pos, table, caches[0], slots, neox)
    pe, k = q.contiguous(), kv[:, R:].unsqueeze(1).contiguous()
    ops.rope_inplace(pe, k, pos, table, is_neox=neox)
    ops.mla_reshape_and_cache(ops.rmsnorm(kv[:, :R], w, 1e-6), k.squeeze(1), caches[1],
                              slots)
    assert torch.equal(got, pe)
    assert torch.equal(caches[0].view(torch.uint8), caches[1].view(torch.uint8))
    args = (w, 1e-6, pos, table, caches[0], slots, neox)
    assert ops.mla_rope_and_cache(q.float(), kv, *args) is None
    assert ops.mla_rope_and_cache(q[..., :DR - 8], kv, *args) is None
    assert ops.mla_rope_and_cache(q, kv[:, 1:], *args) is None


@pytest.mark.parametrize("M,K,R,DR", [(17, 7168, 512, 64), (40, 7168, 512, 64),
                                      (64, 7168, 512, 64), (33, 8192, 64, 16),
                                      (70, 7168, 1544, 128), (20, 16384, 512, 64)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("neox", [False, True])
def test_linear_mla_rope_and_cache(M, K, R, DR, fp8, neox):
    """The same bits as the product and mla_rope_and_cache: parts are added in one
    order. Infinities of x and a token without a slot included."""
    g = torch.Generator(device="cuda").manual_seed(M + K)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    x, kv_w = rand(M, K + 8)[:, :K], rand(R + DR, K) * K ** -0.5
    q, w = rand(M, 3, DR + 32)[..., 32:], rand(R)
    x[3, 5] = float("inf")
    table = torch.randn(90, DR, generator=g, device="cuda")
    pos = torch.randint(0, 90, (M,), generator=g, device="cuda", dtype=torch.int32)
    slots = torch.randperm(96, generator=g, device="cuda")[:M]
    slots[M // 2] = -1
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    caches = [torch.zeros(6, 16, R + DR, device="cuda").to(dt) for _ in range(2)]
    args = lambda c: (w, 1e-6, pos, table, c, slots, neox)
    assert ops.product_has_parts(M, kv_w)
    got = ops.linear_mla_rope_and_cache(x, kv_w, q, *args(caches[0]))
    want = ops.mla_rope_and_cache(q, ops.linear(x, kv_w), *args(caches[1]))
    assert torch.equal(got, want)
    assert torch.equal(caches[0].view(torch.uint8), caches[1].view(torch.uint8))
    run = lambda x=x, kv_w=kv_w, q=q: ops.linear_mla_rope_and_cache(
        x, kv_w, q, *args(caches[0]))
    assert run(x=x[:4], q=q[:4]) is None and run(x=x[:-1]) is None
    assert run(x=x.float()) is None and run(kv_w=kv_w.float()) is None
    assert run(kv_w=kv_w[:-8]) is None and run(q=q.float()) is None
    assert run(x=rand(M, K + 4)[:, 4:]) is None              # rows at odd places
    assert run(kv_w=kv_w.clone().requires_grad_()) is None


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("H,BS,ctxs", [
    (64, 32, [257, 31, 32, 33, 1, 64, 65, 0, 96]),  # ends of tiles of 32, none
    (33, 16, [1000]),                               # heads past the last one
    (100, 64, [300, 129, 4000]),                    # two workgroups, one part full
    (128, 32, [9000, 1, 290]),                      # many runs of one sequence
    (128, 16, [260] + [90, 13, 200] * 50),          # runs that meet sequences
    (64, 32, [20, 255]),                            # a workgroup a sequence
    (16, 32, [3000, 0, 65]),                        # tiles of 64: the same deal
])
def test_mla_decode_tiles_and_runs(H, BS, ctxs, kv):
    """Edges of tiles, runs and sequences; slots past a sequence's end hold NaN."""
    B, scale = len(ctxs), 192 ** -0.5
    ql, qp, cache, bt, sl = _setup(B, H, ctxs, BS=BS, seed=7)
    ql, qp = ql * 10, qp * 10  # unit normal: weights of unequal size
    dt = torch.float8_e4m3fn if kv == "fp8" else torch.bfloat16
    cache = cache.to(dt)
    for i, n in enumerate(ctxs):  # what a sequence has not filled
        if n % BS:
            cache[int(bt[i, n // BS]), n % BS:] = float("nan")
    out = ops.mla_paged_attention_decode(ql, qp, cache, bt, sl, scale)
    again = ops.mla_paged_attention_decode(ql, qp, cache, bt, sl, scale)
    assert torch.equal(out, again)
    for i, n in enumerate(ctxs):
        if n == 0:
            assert not out[i].any()
            continue
        pages = bt[i, :(n + BS - 1) // BS].long()
        e = cache[pages].double().flatten(0, 1)[:n]
        p = ((ql[i].double() @ e[:, :512].T + qp[i].double() @ e[:, 512:].T)
             * scale).softmax(-1)
        want = p @ e[:, :512]
        err = (out[i].double() - want).norm() / want.norm()
        # weights and results are rounded to bf16, each by 2^-8 of it at most and by 2^-9.3
        # in the root mean square, which for weights the sum over tokens makes less
        assert err < 2 * 2 ** -9, (i, n, float(err))


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("H,ctxs", [
    (16, [3200, 64, 200]),      # tiles of 64
    (64, [3200, 64, 200]),      # tiles of 32, several runs
    (128, [224, 32, 200]),      # a workgroup a sequence
])
def test_mla_decode_sums_weights_unrounded(H, ctxs, kv):
    """Every 32nd token weighs 1, the others 2^-3 (1 + 0.45 * 2^-7), which is 2^-3 in
    bf16, and only the former have values: their sum is exact, and a sum of rounded
    weights would be 0.0028 short."""
    ql, qp, cache, bt, sl = _setup(len(ctxs), H, ctxs, seed=11)
    one = torch.arange(32, device="cuda") == 5
    cache[..., 512:] = 0
    cache[..., 512] = torch.where(one, 0.0, -1.0)
    cache[:, ~one, :512] = 0
    ql.zero_(), qp.zero_()
    qp[..., 0] = 1
    if kv == "fp8":
        cache = cache.to(torch.float8_e4m3fn)
    p = 2 ** -3 * (1 + 0.45 * 2 ** -7)
    out = ops.mla_paged_attention_decode(ql, qp, cache, bt, sl, -math.log(p)).double()
    for i, n in enumerate(ctxs):
        e = cache[bt[i, :-(-n // 32)].long()].double().flatten(0, 1)[:n]
        w = torch.where(e[:, 512] == 0, 1.0, p).double()
        want = (w @ e[:, :512]) / w.sum()
        # against the rounded result: fp32's own rounding, 1e-6, moves few of a head's 512
        # values over the middle of two bf16 numbers, each by 2^-7, 2e-5 of all
        off = ((out[i] - want.bfloat16().double()) @ want) / (want @ want)
        assert off.abs().max() < 2e-4, (n, off.abs().max().item())


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("scale", [-192 ** -0.5, 0.0, 1e-6, 3.0])
@pytest.mark.parametrize("H,ctxs", [(16, [700, 65]), (64, [3000, 33]), (128, [200, 31])])
def test_mla_decode_scales_of_any_sign(H, ctxs, scale, kv):
    """Scores are multiplied behind their maximum, whose sign the scale has."""
    ql, qp, cache, bt, sl = _setup(len(ctxs), H, ctxs, seed=13)
    if kv == "fp8":
        cache = cache.to(torch.float8_e4m3fn)
    out = ops.mla_paged_attention_decode(ql, qp, cache, bt, sl, scale)
    for i, n in enumerate(ctxs):
        e = cache[bt[i, :-(-n // 32)].long()].double().flatten(0, 1)[:n]
        s = (ql[i].double() @ e[:, :512].T + qp[i].double() @ e[:, 512:].T) * scale
        want = s.softmax(-1) @ e[:, :512]
        err = (out[i].double() - want).norm() / want.norm()
        assert err < 2 * 2 ** -9, (n, float(err))  # as above


@pytest.mark.parametrize("H,first", [(16, 70), (16, 600), (64, 40), (64, 600), (128, 170)])
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
def test_mla_decode_infinities(H, first, kv):
    """Tokens hidden by a score of -inf, whole tiles and runs of them, at either sign of the
    scale; a sequence with +inf and one with NaN are NaN, and no other is. (An fp8 cache has
    no infinity: rows of -448 take weight 0 from a wide query.)"""
    ctxs = [first + 230 if H < 128 else 200, 90, 80, 150]
    ql, qp, cache, bt, sl = _setup(len(ctxs), H, ctxs, seed=17)
    low = -448.0 if kv == "fp8" else float("-inf")
    qp[..., 0] = 2.0 ** 20 if kv == "fp8" else 1.0
    cache[..., 512] = 0
    rows = [cache[bt[i, :-(-n // 32)].long()].flatten(0, 1)[:n] for i, n in enumerate(ctxs)]
    rows[0][:first, 512] = low
    rows[1][50, 512] = -low
    rows[2][7, 100] = float("nan")
    rows[3][140:, 512] = low
    for i, r in enumerate(rows):
        for j in range(0, len(r), 32):
            cache[int(bt[i, j // 32]), :len(r[j:j + 32])] = r[j:j + 32]
    for scale in (192 ** -0.5, -192 ** -0.5):
        q = qp.clone()
        q[..., 0] *= 1 if scale > 0 else -1
        c = cache.to(torch.float8_e4m3fn) if kv == "fp8" else cache
        out = ops.mla_paged_attention_decode(ql, q, c, bt, sl, scale)
        for i, n in enumerate(ctxs):
            e = c[bt[i, :-(-n // 32)].long()].double().flatten(0, 1)[:n]
            s = (ql[i].double() @ e[:, :512].T + q[i].double() @ e[:, 512:].T) * scale
            want = s.softmax(-1) @ e[:, :512]
            if i == 2 or i == 1 and kv == "bf16":
                assert want.isnan().all() and out[i].isnan().all(), (i, scale)
                continue
            err = (out[i].double() - want).norm() / want.norm()
            assert err < 2 * 2 ** -9, (i, scale, float(err))  # as above


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("H", [16, 64, 128])
@pytest.mark.parametrize("B", [64, 65, 256, 257, 321])
def test_mla_decode_many_sequences(B, H, kv):
    """A lane deals one, four or more sequences' tiles; the last ones as the first."""
    ctxs = [(0, 270, 40, 129, 31)[i * i % 5] + i % 3 for i in range(B)]
    ctxs[-1] = 300
    ql, qp, cache, bt, sl = _setup(B, H, ctxs, seed=B)
    if kv == "fp8":
        cache = cache.to(torch.float8_e4m3fn)
    out = ops.mla_paged_attention_decode(ql, qp, cache, bt, sl, 192 ** -0.5)
    for i, n in enumerate(ctxs):
        if n == 0:
            assert not out[i].any()
            continue
        e = cache[bt[i, :-(-n // 32)].long()].double().flatten(0, 1)[:n]
        s = (ql[i].double() @ e[:, :512].T + qp[i].double() @ e[:, 512:].T) * 192 ** -0.5
        want = s.softmax(-1) @ e[:, :512]
        err = (out[i].double() - want).norm() / want.norm()
        assert err < 2 * 2 ** -9, (i, n, float(err))  # as above
