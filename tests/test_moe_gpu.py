"""Grouped-GEMM MoE kernel vs the CPU reference expert loop."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from parallax_amd import ops


def _cpu_moe(x, w_gu, w_down, topk_ids, topk_w):
    T, H = x.shape
    inter = w_gu.shape[1] // 2
    out = torch.zeros(T, H, dtype=torch.float32)
    for t in range(T):
        for j in range(topk_ids.shape[1]):
            e = int(topk_ids[t, j])
            w = float(topk_w[t, j])
            h = x[t].float() @ w_gu[e].float().T
            gate, up = h[:inter], h[inter:]
            act = torch.nn.functional.silu(gate) * up
            out[t] += w * (act @ w_down[e].float().T)
    return out


@pytest.mark.parametrize("T,E,k,H,I", [
    (16, 8, 2, 128, 64),
    (64, 32, 8, 256, 128),
    (3, 4, 2, 64, 64),     # tiny batch
    (128, 4, 1, 128, 192),  # heavy per-expert load (multi-tile segments)
])
def test_moe_forward(T, E, k, H, I):
    torch.manual_seed(0)
    x = (torch.randn(T, H, dtype=torch.bfloat16, device="cuda") * 0.5)
    w_gu = torch.randn(E, 2 * I, H, dtype=torch.bfloat16, device="cuda") * 0.05
    w_down = torch.randn(E, H, I, dtype=torch.bfloat16, device="cuda") * 0.05
    topk_ids = torch.stack(
        [torch.randperm(E, device="cuda")[:k] for _ in range(T)]
    ).long()
    topk_w = torch.rand(T, k, dtype=torch.float32, device="cuda")
    out = ops.fused_moe_forward(x, w_gu, w_down, topk_ids, topk_w)
    expect = _cpu_moe(x.float().cpu(), w_gu.float().cpu(), w_down.float().cpu(),
                      topk_ids.cpu(), topk_w.cpu())
    torch.testing.assert_close(out.float().cpu(), expect, atol=5e-2, rtol=5e-2)


def _quant_rows(x):
    """Emulate the kernel's per-row activation quantization in torch."""
    amax = x.float().abs().amax(dim=-1).clamp_min(1e-8)
    scale = amax / 448.0
    q = (x.float() / scale.unsqueeze(-1)).clamp(-448, 448).to(torch.float8_e4m3fn)
    return q, scale


def _cpu_moe_fp8(x, w_gu_q, w_gu_s, w_dn_q, w_dn_s, topk_ids, topk_w):
    """fp32 emulation of the W8A8 kernel: fp8-quantized operands, fp32
    accumulate, per-row h quantization between the two GEMMs."""
    T, H = x.shape
    inter = w_gu_q.shape[1] // 2
    out = torch.zeros(T, H, dtype=torch.float32)
    xq, xs = _quant_rows(x)
    for t in range(T):
        for j in range(topk_ids.shape[1]):
            e = int(topk_ids[t, j])
            w = float(topk_w[t, j])
            wg = w_gu_q[e].float() * w_gu_s[e].unsqueeze(-1)
            h = (xq[t].float() * xs[t]) @ wg.T
            gate, up = h[:inter], h[inter:]
            act = (torch.nn.functional.silu(gate) * up).to(torch.bfloat16)
            hq, hs = _quant_rows(act.unsqueeze(0))
            wd = w_dn_q[e].float() * w_dn_s[e].unsqueeze(-1)
            out[t] += w * ((hq[0].float() * hs[0]) @ wd.T)
    return out


@pytest.mark.parametrize("T,E,k,H,I", [
    (16, 8, 2, 128, 64),
    (64, 32, 8, 256, 128),
    (3, 4, 2, 64, 64),
])
def test_moe_forward_fp8(T, E, k, H, I):
    """W8A8 kernel vs a torch emulation with identical quantization (tight)
    and vs the unquantized fp32 reference (loose — quantization error)."""
    torch.manual_seed(0)
    x = (torch.randn(T, H, dtype=torch.bfloat16, device="cuda") * 0.5)
    w_gu = torch.randn(E, 2 * I, H, dtype=torch.bfloat16, device="cuda") * 0.05
    w_down = torch.randn(E, H, I, dtype=torch.bfloat16, device="cuda") * 0.05
    topk_ids = torch.stack(
        [torch.randperm(E, device="cuda")[:k] for _ in range(T)]
    ).long()
    topk_w = torch.rand(T, k, dtype=torch.float32, device="cuda")
    q_gu, s_gu = ops.quantize_fp8_weight(w_gu)
    q_dn, s_dn = ops.quantize_fp8_weight(w_down)
    out = ops.fused_moe_forward_fp8(x, q_gu, s_gu, q_dn, s_dn, topk_ids, topk_w)
    emu = _cpu_moe_fp8(x.float().cpu(), q_gu.cpu(), s_gu.cpu(), q_dn.cpu(),
                       s_dn.cpu(), topk_ids.cpu(), topk_w.cpu())
    torch.testing.assert_close(out.float().cpu(), emu, atol=3e-2, rtol=3e-2)
    fp32 = _cpu_moe(x.float().cpu(), w_gu.float().cpu(), w_down.float().cpu(),
                    topk_ids.cpu(), topk_w.cpu())
    rel = (out.float().cpu() - fp32).norm() / fp32.norm().clamp_min(1e-6)
    assert rel < 0.08, f"fp8 path rel error vs fp32 reference {rel:.3f}"


def test_moe_fp8_engine_decode():
    """DeepSeek-V3-class engine with fp8 expert weights decodes through the
    graph-captured path (reduced layer count)."""
    from parallax_amd.models.config import ModelConfig
    from parallax_amd.server.engine import Engine, EngineArgs
    from parallax_amd.server.sampling_params import SamplingParams

    cfg = ModelConfig.from_hf_config({
        "architectures": ["DeepseekV3ForCausalLM"], "model_type": "deepseek_v3",
        "vocab_size": 512, "hidden_size": 256, "num_hidden_layers": 3,
        "num_attention_heads": 8, "num_key_value_heads": 8,
        "intermediate_size": 512, "moe_intermediate_size": 128,
        "n_routed_experts": 16, "num_experts_per_tok": 4, "n_shared_experts": 1,
        "n_group": 4, "topk_group": 2, "routed_scaling_factor": 2.5,
        "norm_topk_prob": True, "first_k_dense_replace": 1,
        "q_lora_rank": 128, "kv_lora_rank": 512, "qk_nope_head_dim": 64,
        "qk_rope_head_dim": 64, "v_head_dim": 64, "rms_norm_eps": 1e-6,
        "rope_theta": 10000.0, "max_position_embeddings": 2048,
    })
    eng = Engine(cfg, EngineArgs(num_kv_blocks=128, moe_weight_dtype="fp8"),
                 random_weights=True)
    out = eng.generate(
        [[1, 2, 3, 4, 5], [7] * 20],
        [SamplingParams(temperature=0.0, max_new_tokens=6, ignore_eos=True)] * 2,
    )
    assert all(len(v) == 6 for v in out.values())


def test_moe_engine_graph_capture():
    """MoE model decodes through the graph-captured path."""
    from parallax_amd.models.config import ModelConfig
    from parallax_amd.server.engine import Engine, EngineArgs
    from parallax_amd.server.sampling_params import SamplingParams

    cfg = ModelConfig(
        architecture="Qwen3MoeForCausalLM", model_type="qwen3_moe",
        vocab_size=512, hidden_size=256, num_layers=2, num_heads=4,
        num_kv_heads=2, head_dim=64, intermediate_size=512,
        moe_intermediate_size=128, num_experts=8, num_experts_per_tok=2,
        max_position_embeddings=2048, eos_token_ids=[],
    )
    eng = Engine(cfg, EngineArgs(num_kv_blocks=128), random_weights=True)
    out = eng.generate(
        [[1, 2, 3, 4, 5], [7] * 20],
        [SamplingParams(temperature=0.0, max_new_tokens=6, ignore_eos=True)] * 2,
    )
    assert eng.graph_runner is not None and len(eng.graph_runner._graphs) > 0
    assert all(len(v) == 6 for v in out.values())


def _experts64(x, gu, dn, ids, w, fp8=False, on_input=False, bias=None,
               limit=0.0, gelu=False):
    """The experts in float64 on the device, one at a time; fp8: operands
    quantised a row before both products."""
    def q8(t):
        s = t.abs().amax(-1, keepdim=True).clamp_min(1e-8) / 448.0
        return (t / s).float().to(torch.float8_e4m3fn).double() * s

    inter = dn.shape[2]
    xd = q8(x.double()) if fp8 else x.double()
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    for e in range(gu.shape[0]):
        t, j = (ids == e).nonzero(as_tuple=True)
        wt = w[t, j].double()[:, None]
        h = xd[t] @ gu[e].double().T
        if on_input:
            h = h * wt
        if bias is not None:
            h = h + bias[e].double()
        g, u = h[:, :inter], h[:, inter:]
        if limit:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            a = (u + 1) * g * torch.sigmoid(1.702 * g)
        elif gelu:
            a = torch.nn.functional.gelu(g, approximate="tanh") * u
        else:
            a = torch.nn.functional.silu(g) * u
        a = q8(a.bfloat16().double()) if fp8 else a
        y = a @ dn[e].double().T
        out.index_add_(0, t, y if on_input else y * wt)
    return out


@pytest.mark.parametrize("T,E,k,H,I,fp8", [
    # tiles of 32 rows
    (1, 3, 1, 32, 32, False),       # less than a stage of the contraction
    (40, 5, 2, 96, 96, False),      # its last stage partly filled
    # of 64
    (300, 2, 1, 160, 352, False),   # several tiles an expert, odd features
    (450, 3, 2, 320, 288, False),   # and remainders of every height
    (40, 5, 2, 96, 64, True),
    (700, 6, 2, 224, 192, True),
    # of 256
    (5000, 9, 2, 64, 32, False),    # choices counted in parts
])
def test_moe_tiles(T, E, k, H, I, fp8):
    """Tile heights, remainders of rows, features and contraction, experts
    without a token and choices of another rank's expert (id E). bf16: h is
    rounded once, 2^-9 relative, so the error's norm stays below 2^-8 of the
    result's; fp8: h values next to a rounding edge move by one e4m3 step
    (2^-3) where the fp32 sums differ in their last bits: below 2 %."""
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    gu = (torch.randn(E, 2 * I, H, generator=g, device="cuda") * H ** -0.5).bfloat16()
    dn = (torch.randn(E, H, I, generator=g, device="cuda") * I ** -0.5).bfloat16()
    ids = torch.rand(T, E + 1, generator=g, device="cuda")
    ids[:, E // 2] = -1                       # an expert that nobody chooses
    ids = ids.topk(k, dim=-1).indices
    w = torch.rand(T, k, generator=g, device="cuda")
    if fp8:
        qg, sg = ops.quantize_fp8_weight(gu)
        qd, sd = ops.quantize_fp8_weight(dn)
        got = ops.fused_moe_forward_fp8(x, qg, sg, qd, sd, ids, w)
        want = _experts64(x, qg.double() * sg[..., None], qd.double() * sd[..., None],
                          ids, w, fp8=True)
        assert (got - want).norm() < 2e-2 * want.norm()
        return
    for kw in ({}, {"on_input": True}, {"limit": 7.0}, {"gelu": True}):
        bias = (torch.randn(E, 2 * I, generator=g, device="cuda").bfloat16()
                if "limit" in kw else None)
        got = ops.fused_moe_forward(
            x, gu, dn, ids, w, activation="gelu" if kw.get("gelu") else "silu",
            limit=kw.get("limit", 0.0), bias_gate_up=bias,
            weight_on_input=kw.get("on_input", False))
        want = _experts64(x, gu, dn, ids, w, bias=bias, **kw)
        assert (got - want).norm() < 2 ** -8 * want.norm()
    assert ops.fused_moe_forward(x[:0], gu, dn, ids[:0], w[:0]).shape == (0, H)


@pytest.mark.parametrize("T,E,k,H", [
    (41, 5, 2, 96),         # rows that do not fill the last workgroup
    (47, 5, 2, 2080),       # longer than its threads' first pass
    (5001, 5, 2, 96),       # beside choices that are counted in parts
    (47, 8200, 2, 32),      # counters of experts that do not fit the LDS
])
def test_moe_rows_quantised_beside_the_routing(T, E, k, H):
    """Rows of other magnitudes and one of zeros: were every value of a row's h moved by
    one e4m3 step, its result would move by 2^-3 at most."""
    g = torch.Generator(device="cuda").manual_seed(T + H)
    x = torch.randn(T, H, generator=g, device="cuda")
    x = (x * 2.0 ** (torch.arange(T, device="cuda") % 13 - 6)[:, None]).bfloat16()
    x[3] = 0
    gu = (torch.randn(E, 128, H, generator=g, device="cuda") * H ** -0.5).bfloat16()
    dn = (torch.randn(E, H, 64, generator=g, device="cuda") / 8).bfloat16()
    ids = torch.rand(T, min(E, 40), generator=g, device="cuda").topk(k, dim=-1).indices
    ids = ids + (E - min(E, 40))
    w = torch.rand(T, k, generator=g, device="cuda")
    qg, sg = ops.quantize_fp8_weight(gu)
    qd, sd = ops.quantize_fp8_weight(dn)
    got = ops.fused_moe_forward_fp8(x, qg, sg, qd, sd, ids, w)
    first = E - min(E, 40)  # the oracle goes through the experts that are chosen
    want = _experts64(x, (qg[first:].double() * sg[first:, :, None]),
                      qd[first:].double() * sd[first:, :, None], ids - first, w, fp8=True)
    assert ((got - want).norm(dim=1) <= 2 ** -3 * want.norm(dim=1)).all()


@pytest.mark.parametrize("H,I,fp8", [
    (96, 96, False),      # a stage and a half, then half a stage
    (704, 544, False),    # 11 and 8.5 stages; 544 features: blocks cut by the end
    (32, 32, False),      # less than a stage
    (160, 192, True),
    (896, 64, True),
])
def test_moe_rows_of_large_tiles(H, I, fp8):
    """Tiles of 256 rows at the edges of their steps of 64: 1 .. 512 rows an expert.
    Every row on its own: a row that is wrong does not hide among the others. bf16 as in
    test_moe_tiles, 2^-7 for a row's spread; fp8: were every value of a row's h moved by
    one e4m3 step, 2^-3 of it, the row's result would move by as much of its norm."""
    rows = [1, 64, 65, 128, 0, 129, 192, 193, 256, 257, 511, 512, 3000]
    E, n = len(rows) + 1, sum(rows)
    g = torch.Generator(device="cuda").manual_seed(H)
    owner = torch.repeat_interleave(torch.arange(len(rows)), torch.tensor(rows))
    owner = owner[torch.randperm(n, generator=torch.Generator().manual_seed(1))]
    owner = torch.cat([owner, owner.new_full((16384 - n,), E)])  # of another rank
    ids = owner.view(-1, 2).cuda()
    T = ids.shape[0]
    assert 16384 // E > 450                     # tiles of 256 rows by the rule
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    gu = (torch.randn(E, 2 * I, H, generator=g, device="cuda") * H ** -0.5).bfloat16()
    dn = (torch.randn(E, H, I, generator=g, device="cuda") * I ** -0.5).bfloat16()
    w = 0.5 + 0.5 * torch.rand(T, 2, generator=g, device="cuda")  # no choice is small
    if fp8:
        qg, sg = ops.quantize_fp8_weight(gu)
        qd, sd = ops.quantize_fp8_weight(dn)
        for kw in ({}, {"limit": 7.0}, {"gelu": True}):
            got = ops.fused_moe_forward_fp8(
                x, qg, sg, qd, sd, ids, w, limit=kw.get("limit", 0.0),
                activation="gelu" if kw.get("gelu") else "silu")
            want = _experts64(x, qg.double() * sg[..., None],
                              qd.double() * sd[..., None], ids, w, fp8=True, **kw)
            err = (got - want).norm(dim=1)
            assert (err <= 2 ** -3 * want.norm(dim=1) + 1e-30).all()
            assert (got - want).norm() < 2e-2 * want.norm()
        return
    bias = torch.randn(E, 2 * I, generator=g, device="cuda").bfloat16()
    for kw in ({}, {"on_input": True}, {"limit": 7.0, "bias": bias}, {"gelu": True}):
        got = ops.fused_moe_forward(
            x, gu, dn, ids, w, activation="gelu" if kw.get("gelu") else "silu",
            limit=kw.get("limit", 0.0), bias_gate_up=kw.get("bias"),
            weight_on_input=kw.get("on_input", False))
        want = _experts64(x, gu, dn, ids, w, **kw)
        err = (got - want).norm(dim=1)
        assert (err <= 2 ** -7 * want.norm(dim=1) + 1e-30).all()


@pytest.mark.parametrize("T", [40, 300, 5000])   # tiles of 32, 64 and 256 rows
def test_moe_infinities(T):
    """An infinite activation reaches its own row, an infinite weight the rows of its
    expert; all others keep their bits. H and I end within a stage."""
    g = torch.Generator(device="cuda").manual_seed(T)
    E, H, I = 5, 96, 96
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    gu = (torch.randn(E, 2 * I, H, generator=g, device="cuda") * H ** -0.5).bfloat16()
    dn = (torch.randn(E, H, I, generator=g, device="cuda") * I ** -0.5).bfloat16()
    ids = torch.randint(0, E, (T, 1), generator=g, device="cuda")
    ids[:2, 0] = 0
    w = 0.5 + torch.rand(T, 1, generator=g, device="cuda")
    want = ops.fused_moe_forward(x, gu, dn, ids, w)
    x[1, H - 1] = gu[3, 7, H - 1] = dn[4, 5, I - 1] = float("inf")
    got = ops.fused_moe_forward(x, gu, dn, ids, w)
    e = ids[:, 0]
    assert not got[1].isfinite().all() and not got[e == 3].isfinite().any()
    assert not got[e == 4][:, 5].isfinite().any()
    got[:, 5] = torch.where(e == 4, want[:, 5], got[:, 5])
    same = e != 3
    same[1] = False
    assert torch.equal(got[same], want[same])


@pytest.mark.parametrize("fp8", [False, True])
def test_moe_many_choices_within_a_fixed_workspace(fp8):
    """The down product and its combine go over the output features in slabs once a
    row a choice would take more than 256 MB: here two, the second narrower. The
    same sums as of a few tokens at a time, in the same order."""
    g = torch.Generator(device="cuda").manual_seed(2)
    T, E, k, H, I = 4096, 5, 8, 2592, 64
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    w_gu = torch.randn(E, 2 * I, H, generator=g, device="cuda") * H ** -0.5
    w_dn = torch.randn(E, H, I, generator=g, device="cuda") * I ** -0.5
    ids = torch.randint(-1, E, (T, k), generator=g, device="cuda")
    wts = torch.rand(T, k, generator=g, device="cuda")
    if fp8:
        w_gu, s_gu = ops.quantize_fp8_weight(w_gu)
        w_dn, s_dn = ops.quantize_fp8_weight(w_dn)
        run = lambda s: ops.fused_moe_forward_fp8(x[s], w_gu, s_gu, w_dn, s_dn,
                                                  ids[s], wts[s])
    else:
        w_gu, w_dn = w_gu.bfloat16(), w_dn.bfloat16()
        run = lambda s: ops.fused_moe_forward(x[s], w_gu, w_dn, ids[s], wts[s])
    want = torch.cat([run(slice(i, i + 512)) for i in range(0, T, 512)])
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    out = run(slice(0, T))
    # besides it x in fp8, h in bf16 and fp8, scales, the order: below 32 MB
    assert torch.cuda.max_memory_allocated() - before < (
        (256 << 20) + out.numel() * 4 + (32 << 20))
    assert torch.equal(out, want)


@pytest.mark.parametrize("E", [8192, 8193, 20000])
@pytest.mark.parametrize("T", [3, 70])
def test_moe_many_experts(E, T):
    """More experts than their counters have room in LDS; most are chosen by none,
    some by many, the first and the last by some."""
    g = torch.Generator(device="cuda").manual_seed(E)
    H, I, k = 64, 32, 4
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    w_gu = (torch.randn(E, 2 * I, H, generator=g, device="cuda") * 0.1).bfloat16()
    w_dn = (torch.randn(E, H, I, generator=g, device="cuda") * 0.2).bfloat16()
    ids = torch.randint(0, E, (T, k), generator=g, device="cuda")
    ids[:, 0] = torch.tensor([0, E - 1, 5000], device="cuda").repeat(24)[:T]
    ids[1, 2] = E
    wts = torch.rand(T, k, generator=g, device="cuda")
    out = ops.fused_moe_forward(x, w_gu, w_dn, ids, wts)
    wts[1, 2], ids[1, 2] = 0, 0
    used, local = ids.cpu().unique(return_inverse=True)
    want = _cpu_moe(x.cpu(), w_gu[used.cuda()].cpu(), w_dn[used.cuda()].cpu(), local,
                    wts.cpu())
    # h is rounded to bf16: 2^-9 of sums of |h w| < 4 weights * 32 * |h| 3 * |w| 0.9
    torch.testing.assert_close(out.cpu(), want, atol=0.05, rtol=1e-2)


@pytest.mark.parametrize("T,E,k,H,I,fp8", [
    (1, 3, 1, 64, 64, False),         # one stage along K, three waves without any
    (32, 3, 1, 192, 128, False),      # experts of several times eight rows
    (4, 6, 8, 320, 448, False),       # a token that chooses an expert twice
    (8, 40, 4, 2112, 192, False),     # a size that the kernels for more choices take
    (5, 20, 4, 4032, 192, False),     # 16 features a workgroup
    (4, 128, 8, 2048, 128, False),    # most experts met once
    (2, 9, 8, 2048, 768, False),
    (1, 2, 1, 128, 128, True),
    (16, 3, 1, 384, 256, True),
    (2, 30, 8, 2176, 640, True),
])
def test_moe_few(T, E, k, H, I, fp8):
    """At most 32 choices (fp8: 16): every token on its own, bounds as in the tests of
    tiles. Choices of other ranks' experts, a token without any other."""
    g = torch.Generator(device="cuda").manual_seed(T + H)
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    gu = (torch.randn(E, 2 * I, H, generator=g, device="cuda") * H ** -0.5).bfloat16()
    dn = (torch.randn(E, H, I, generator=g, device="cuda") * I ** -0.5).bfloat16()
    ids = torch.randint(0, E, (T, k), generator=g, device="cuda")
    if T > 2:
        ids[1], ids[2, 0] = E, -1
    if k > E:
        ids[0, :2] = 4
    w = 0.5 + 0.5 * torch.rand(T, k, generator=g, device="cuda")
    bias = torch.randn(E, 2 * I, generator=g, device="cuda").bfloat16()
    if fp8:
        (qg, sg), (qd, sd) = ops.quantize_fp8_weight(gu), ops.quantize_fp8_weight(dn)
        gu, dn = qg.double() * sg[..., None], qd.double() * sd[..., None]
    for kw in ({}, {"limit": 7.0}, {"gelu": True}) + (
            () if fp8 else ({"on_input": True}, {"bias": bias})):
        act = "gelu" if kw.get("gelu") else "silu"
        if fp8:
            got = ops.fused_moe_forward_fp8(x, qg, sg, qd, sd, ids, w, activation=act,
                                            limit=kw.get("limit", 0.0))
        else:
            got = ops.fused_moe_forward(
                x, gu, dn, ids, w, activation=act, limit=kw.get("limit", 0.0),
                bias_gate_up=kw.get("bias"), weight_on_input=kw.get("on_input", False))
        want = _experts64(x, gu, dn, ids, w, fp8=fp8, **kw)
        err = (got - want).norm(dim=1)
        assert (err <= (2 ** -3 if fp8 else 2 ** -7) * want.norm(dim=1) + 1e-30).all()
        assert (got - want).norm() < (2e-2 if fp8 else 2 ** -8) * want.norm()


@pytest.mark.parametrize("n,E,H,I,fp8,takes", [
    (32, 128, 2048, 768, False, True),    # an expert a choice, a workgroup a CU
    (32, 32, 2048, 1024, False, True), (16, 16, 1024, 512, False, True),
    (8, 256, 7168, 2048, True, True), (16, 256, 7168, 2048, True, False),
    (32, 128, 256, 768, False, False),    # 32 workgroups for all of the second launch
    (32, 3, 256, 768, False, True),       # of three experts
    (24, 64, 4480, 1280, False, False),   # 24 workgroups beyond a round
    (24, 64, 4096, 1280, False, True),
    (8, 128, 256, 3072, False, True), (9, 128, 256, 3072, False, False),  # but up to eight
    (33, 3, 2048, 768, False, False), (17, 3, 2048, 768, True, False),
    (8, 8, 2048, 160, True, False), (8, 8, 96, 128, False, False),  # K in no whole stages
    (1, 1, 64, 64, False, True),
])
def test_moe_few_is_taken_where_it_is_faster(n, E, H, I, fp8, takes):
    assert ops._require_ext("moe_few_takes").moe_few_takes(n, E, H, I, fp8) == takes


def test_moe_few_infinities_and_graph():
    """An infinite weight reaches the results of its expert's rows alone; a replay takes
    the choices of then."""
    g = torch.Generator(device="cuda").manual_seed(3)
    T, E, k, H, I = 6, 5, 2, 192, 192
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    gu = (torch.randn(E, 2 * I, H, generator=g, device="cuda") * H ** -0.5).bfloat16()
    dn = (torch.randn(E, H, I, generator=g, device="cuda") * I ** -0.5).bfloat16()
    ids = torch.tensor([[0, 1], [1, 2], [2, 3], [3, 0], [1, 0], [2, 0]], device="cuda")
    w = 0.5 + torch.rand(T, k, generator=g, device="cuda")
    want = ops.fused_moe_forward(x, gu, dn, ids, w)
    gu[4, 3, H - 1] = dn[4, 5, I - 1] = dn[3, 7, 0] = float("inf")
    got = ops.fused_moe_forward(x, gu, dn, ids, w)
    hit = (ids == 3).any(1)
    assert not got[hit, 7].isfinite().any()
    got[hit, 7] = want[hit, 7]
    assert torch.equal(got, want)
    dn[3, 7, 0] = gu[4, 3, H - 1] = dn[4, 5, I - 1] = 0
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = ops.fused_moe_forward(x, gu, dn, ids, w)
    for step in range(3):
        ids.copy_((ids + 1) % E)
        x.mul_(-0.5)
        eager = ops.fused_moe_forward(x, gu, dn, ids, w)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


@pytest.mark.parametrize("k", [1, 2, 3, 4, 7, 8, 9, 17, 70])
def test_moe_combine_leaves_out_rows_nobody_wrote(k):
    """Choices are added up two, four or eight at a time, and looked at 64 at a time.
    Those of no expert have rows that nothing writes, here over memory that held NaN; a
    token of such choices only is zero."""
    g = torch.Generator(device="cuda").manual_seed(k)
    T, E, H, I = 40, 20, 320, 64
    x = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    gu = (torch.randn(E, 2 * I, H, generator=g, device="cuda") * H ** -0.5).bfloat16()
    dn = (torch.randn(E, H, I, generator=g, device="cuda") * I ** -0.5).bfloat16()
    ids = torch.randint(-1, E + 1, (T, k), generator=g, device="cuda")
    ids[3], ids[4], ids[4, -1] = -1, E, 0
    w = 0.5 + 0.5 * torch.rand(T, k, generator=g, device="cuda")
    want = _experts64(x, gu, dn, ids, w)
    poison = [torch.full((T * k, H), float("nan"), device="cuda") for _ in range(4)]
    del poison
    got = ops.fused_moe_forward(x, gu, dn, ids, w)
    assert not got[3].any() and not got[~((ids >= 0) & (ids < E)).any(1)].any()
    assert ((got - want).norm(dim=1) <= 2 ** -7 * want.norm(dim=1) + 1e-30).all()


def test_moe_combine_reads_rows_of_local_experts_alone():
    """With all experts on other ranks eight choices a token cost no more than what one
    does but for their ids: 134 MB of zeros, where 1,074 MB of rows would be read."""
    T, E, H, I = 16384, 4, 2048, 64
    x = torch.zeros(T, H, dtype=torch.bfloat16, device="cuda")
    gu = torch.zeros(E, 2 * I, H, dtype=torch.bfloat16, device="cuda")
    dn = torch.zeros(E, H, I, dtype=torch.bfloat16, device="cuda")

    def fastest(k):
        ids = torch.full((T, k), E, device="cuda")
        w = torch.ones(T, k, device="cuda")
        at = [torch.cuda.Event(enable_timing=True) for _ in range(21)]
        for e in at:
            e.record()
            assert e is at[-1] or ops.fused_moe_forward(x, gu, dn, ids, w).shape == (T, H)
        torch.cuda.synchronize()
        return min(a.elapsed_time(b) for a, b in zip(at, at[1:]))

    fastest(1)
    assert fastest(8) < 2.5 * fastest(1)
