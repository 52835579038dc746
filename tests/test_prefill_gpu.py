"""MFMA prefill attention kernel vs fp32 reference (asymmetric random data —
catches operand/output transposes per the CDNA guide's methodology)."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from parallax_amd import ops
from parallax_amd.ops import reference as ref


def _setup(query_lens, seq_lens, Hq, Hk, D, BS=32, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    B = len(query_lens)
    max_blocks = (max(seq_lens) + BS - 1) // BS
    NB = B * max_blocks + 1
    kc = torch.randn(NB, Hk, BS, D, generator=g, dtype=torch.bfloat16, device="cuda")
    vc = torch.randn(NB, Hk, D, BS, generator=g, dtype=torch.bfloat16, device="cuda")
    bt = (
        torch.arange(B * max_blocks, dtype=torch.int32, device="cuda").reshape(B, max_blocks)
        + 1
    )
    T = sum(query_lens)
    q = torch.randn(T, Hq, D, generator=g, dtype=torch.bfloat16, device="cuda")
    return q, kc, vc, bt, torch.tensor(seq_lens, dtype=torch.int32, device="cuda"), \
        torch.tensor(query_lens, dtype=torch.int32, device="cuda")


def _run(q, kc, vc, bt, sl, ql, D, **kw):
    scale = 1.0 / math.sqrt(D)
    out = ops.prefill_attention(q, kc, vc, bt, sl, ql, scale, **kw)
    expect = ref.prefill_attention(
        q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt.cpu(),
        sl.cpu(), ql.cpu(), scale,
        **{k: (v.cpu() if torch.is_tensor(v) else v) for k, v in kw.items()},
    )
    torch.testing.assert_close(
        out.float().cpu(), expect.float().cpu(), atol=4e-2, rtol=4e-2
    )


@pytest.mark.parametrize("D", [128, 64])
def test_prefill_no_prefix(D):
    # pure prefill: seq_len == query_len, varlen batch incl. non-multiple-of-32
    q, kc, vc, bt, sl, ql = _setup([64, 33, 100], [64, 33, 100], 8, 2, D)
    _run(q, kc, vc, bt, sl, ql, D)


def test_prefill_with_prefix():
    # chunked prefill: earlier tokens already cached (prefix 96 and 32)
    q, kc, vc, bt, sl, ql = _setup([32, 64], [128, 96], 4, 4, 128)
    _run(q, kc, vc, bt, sl, ql, 128)


def test_prefill_single_token_rows():
    q, kc, vc, bt, sl, ql = _setup([1, 1, 5], [40, 1, 5], 8, 2, 128)
    _run(q, kc, vc, bt, sl, ql, 128)


def test_prefill_long():
    q, kc, vc, bt, sl, ql = _setup([1024], [1024], 4, 4, 128, seed=3)
    _run(q, kc, vc, bt, sl, ql, 128)


def test_prefill_sliding_window():
    q, kc, vc, bt, sl, ql = _setup([128], [256], 8, 2, 128, seed=4)
    _run(q, kc, vc, bt, sl, ql, 128, sliding_window=64)


def test_prefill_softcap_sinks():
    q, kc, vc, bt, sl, ql = _setup([64], [64], 8, 2, 128, seed=5)
    sinks = torch.randn(8, dtype=torch.float32, device="cuda")
    _run(q, kc, vc, bt, sl, ql, 128, softcap=20.0, sinks=sinks)


def test_prefill_engine_parity_gpu_vs_cpu():
    """Greedy tokens from the GPU engine (HIP prefill+decode, bf16) match the
    CPU fp32 engine on a tiny model (loose but end-to-end)."""
    from parallax_amd.models.config import ModelConfig
    from parallax_amd.server.engine import Engine, EngineArgs
    from parallax_amd.server.sampling_params import SamplingParams
    from parallax_amd.models import get_model_class

    cfg = ModelConfig(
        architecture="LlamaForCausalLM", vocab_size=256, hidden_size=512,
        num_layers=2, num_heads=4, num_kv_heads=2, head_dim=128,
        intermediate_size=1024, max_position_embeddings=2048, eos_token_ids=[],
    )
    prompts = [[3, 17, 42, 99, 5] * 9, [7] * 40]  # 45 and 40 tokens
    sp = [SamplingParams(temperature=0.0, max_new_tokens=4, ignore_eos=True)] * 2

    eng_gpu = Engine(cfg, EngineArgs(num_kv_blocks=256), random_weights=True)
    out_gpu = list(eng_gpu.generate(prompts, sp).values())

    import parallax_amd.parallel.comm as comm_mod
    ctx = comm_mod.get_comm()
    cpu_ctx = comm_mod.CommContext(
        world_size=1, rank=0, pp_size=1, tp_size=1, pp_rank=0, tp_rank=0,
        device=torch.device("cpu"),
    )
    eng_cpu = Engine(
        cfg, EngineArgs(num_kv_blocks=256, dtype=torch.float32), comm=cpu_ctx,
        random_weights=True,
    )
    comm_mod.set_comm(ctx)
    out_cpu = list(eng_cpu.generate(prompts, sp).values())
    # random init + bf16-vs-fp32: expect identical argmax on a tiny model
    assert out_gpu == out_cpu


@pytest.mark.parametrize("Hq,Hk,D,BS,fp8,kw", [
    (4, 4, 128, 16, False, {}),                       # one row an item
    (14, 2, 64, 32, False, {}),                       # rows cut by a tile's edge
    (16, 1, 128, 64, False, {"sliding_window": 70}),
    (8, 2, 128, 8, False, {"softcap": 30.0}),         # general page sizes
    (8, 2, 64, 24, False, {}),
    (8, 1, 128, 16, True, {}),
    (8, 2, 64, 40, True, {"sliding_window": 33}),
])
def test_prefill_items_pages_and_splits(Hq, Hk, D, BS, fp8, kw):
    """Portions around the 128-item and 64-key tiles, requests of one row, and
    (few items, long prefix) keys split over workgroups. Slots past the end of
    a sequence hold NaN. Weights and results are rounded to bf16 once each:
    an error of at most 2 * 2^-9 * max |v|, max |v| < 5.2 here."""
    per = max(1, 128 // (Hq // Hk))
    for ql, pre in (([per, 1, per + 1], [0, 63, 64]), ([3], [2100])):
        sl = [a + b for a, b in zip(ql, pre)]
        q, kc, vc, bt, slt, qlt = _setup(ql, sl, Hq, Hk, D, BS=BS, seed=len(ql))
        if fp8:
            kc, vc = (t.to(torch.float8_e4m3fn) for t in (kc, vc))
        ref_k, ref_v = kc.float(), vc.float()
        for i, n in enumerate(sl):
            if n % BS and not fp8:
                page = int(bt[i, n // BS])
                kc[page, :, n % BS:] = float("nan")
                vc[page, :, :, n % BS:] = float("nan")
        out = ops.prefill_attention(q, kc, vc, bt, slt, qlt, D ** -0.5, **kw)
        want = ref.prefill_attention(
            q.float().cpu(), ref_k.cpu(), ref_v.cpu(), bt.cpu(), slt.cpu(),
            qlt.cpu(), D ** -0.5, **kw)
        torch.testing.assert_close(out.float().cpu(), want, atol=2.1e-2, rtol=0)


@pytest.mark.parametrize("D,Hq,Hk,ql,pre,window,scale", [
    (64, 64, 8, 512, 0, 128, 0.125),       # rows 63 modulo 64: first tile unseen
    (64, 14, 2, 512, 0, 128, 0.125),       # rows cut by a tile's edge
    (64, 16, 16, 2300, 0, 2047, 0.125),
    (64, 8, 1, 261, 0, 127, 0.1),
    (64, 8, 8, 261, 30, 65, 80 ** -0.5),
    (128, 8, 2, 300, 0, 100, 1 / 12),
    (128, 8, 8, 200, 37, 65, 1 / 128),
    (64, 14, 2, 40, 4607, -1, 0.125),      # the last split begins at the diagonal
    (64, 14, 2, 40, 4607, 700, 0.125),
    (64, 8, 2, 200, 50, 70, -0.125),
    (64, 8, 2, 200, 50, 70, 0.0),
    (128, 8, 2, 40, 2000, 70, 0.0),
])
@pytest.mark.parametrize("sinks", [False, True])
def test_prefill_rows_whose_first_tile_is_hidden(D, Hq, Hk, ql, pre, window, scale,
                                                 sinks):
    """Items that see no key of the first tile their wave computes, by a window or
    by a split of the keys, for scales whose product with a hidden score rounds
    either way. Tolerance as above; sinks take weight away only."""
    q, kc, vc, bt, sl, qlt = _setup([ql], [pre + ql], Hq, Hk, D, seed=ql)
    sk = torch.linspace(-2, 2, Hq, device="cuda") if sinks else None
    out = ops.prefill_attention(q, kc, vc, bt, sl, qlt, scale,
                                sliding_window=window, sinks=sk)
    assert bool(out.isfinite().all())
    want = ref.prefill_attention(
        q.float().cpu(), kc.float().cpu(), vc.float().cpu(), bt.cpu(), sl.cpu(),
        qlt.cpu(), scale, sliding_window=window, sinks=sk.cpu() if sinks else None)
    torch.testing.assert_close(out.float().cpu(), want, atol=2.1e-2, rtol=0)


@pytest.mark.parametrize("fp8", [False, True])
def test_prefill_portion_without_context(fp8):
    """A request whose context is shorter than its portion, or empty, reads no page
    for the rows before it (its table row holds a page that is not there); the other
    requests are right."""
    q, kc, vc, bt, sl, ql = _setup([40, 70, 33], [64, 70, 33], 8, 2, 64, seed=11)
    if fp8:
        kc, vc = (t.to(torch.float8_e4m3fn) for t in (kc, vc))
    bt[1], sl[1] = -1, 0
    out = ops.prefill_attention(q, kc, vc, bt, sl, ql, 0.125)
    keep = torch.cat([torch.arange(40), torch.arange(110, 143)]).cuda()
    pick = torch.tensor([0, 2], device="cuda")
    want = ref.prefill_attention(q[keep].float(), kc.float(), vc.float(), bt[pick],
                                 sl[pick], ql[pick], 0.125)
    torch.testing.assert_close(out[keep].float(), want, atol=2.1e-2, rtol=0)


@pytest.mark.parametrize("Hq,Hk,D,BS,fp8,window", [
    (8, 2, 128, 32, False, -1),
    (8, 2, 128, 16, False, 200),
    (4, 4, 128, 64, False, 300),
    (16, 2, 128, 24, False, -1),       # general page size
    (16, 2, 128, 32, True, -1),
    (8, 2, 128, 64, True, 200),
    (16, 2, 64, 16, False, 200),
    (16, 2, 64, 32, True, -1),
])
def test_prefill_contexts_of_few_tiles(Hq, Hk, D, BS, fp8, window):
    """Contexts of every number of 64-key tiles from one to ten, ending at a tile's
    edge and beside it: turns of pairs of tiles, the first and last turn alone, tiles
    that the diagonal or the window cuts on either side of whole ones. Slots past the
    end hold NaN. Tolerance as above."""
    sl = sorted({64 * n + d for n in range(1, 11) for d in (-1, 0, 1, 32)})
    ql = [min(n, 1 + 7 * i % 70) for i, n in enumerate(sl)]
    q, kc, vc, bt, slt, qlt = _setup(ql, sl, Hq, Hk, D, BS=BS, seed=D + BS)
    if fp8:
        kc, vc = (t.to(torch.float8_e4m3fn) for t in (kc, vc))
    ref_k, ref_v = kc.float(), vc.float()
    for i, n in enumerate(sl):
        if n % BS and not fp8:
            page = int(bt[i, n // BS])
            kc[page, :, n % BS:] = float("nan")
            vc[page, :, :, n % BS:] = float("nan")
    out = ops.prefill_attention(q, kc, vc, bt, slt, qlt, D ** -0.5,
                                sliding_window=window)
    want = ref.prefill_attention(
        q.float().cpu(), ref_k.cpu(), ref_v.cpu(), bt.cpu(), slt.cpu(), qlt.cpu(),
        D ** -0.5, sliding_window=window)
    torch.testing.assert_close(out.float().cpu(), want, atol=2.1e-2, rtol=0)
