"""Decode attention that rotates and stores the step's token itself: the same bits, in
the result and in the cache, as rope_and_cache and paged_attention_decode apart."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from parallax_amd import ops


def _inputs(Hq, Hk, D, BS, lens, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*s):
        return torch.randn(*s, generator=g, device="cuda").bfloat16()

    B = len(lens)
    qkv = randn(B, (Hq + 2 * Hk) * D)
    q, k, v = (t.view(B, -1, D) for t in qkv.split([Hq * D, Hk * D, Hk * D], 1))
    counts = [(n + BS - 1) // BS for n in lens]
    ids = torch.randperm(sum(counts) + 1, generator=g, device="cuda").tolist()
    bt = torch.zeros(B, max(counts), dtype=torch.int32)
    at = 0
    for i, c in enumerate(counts):
        bt[i, :c] = torch.tensor(ids[at:at + c], dtype=torch.int32)
        at += c
    slots = [int(bt[i, (n - 1) // BS]) * BS + (n - 1) % BS for i, n in enumerate(lens)]
    kc, vc = randn(len(ids), Hk, BS, D), randn(len(ids), Hk, D, BS)
    cs = torch.randn(max(lens) + 5, D, generator=g, device="cuda")
    sl = torch.tensor(lens, dtype=torch.int32, device="cuda")
    # the place in the rope table need not be the place in the cache
    pos = (sl + 3).contiguous()
    slots = torch.tensor(slots, dtype=torch.int64, device="cuda")
    return q, k, v, kc, vc, pos, cs, slots, bt.cuda(), sl


SHORT = [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 513, 600, 1000]
LONG = [5000, 1, 33, 4096, 128, 2047, 3000]


@pytest.mark.parametrize("Hq,Hk,D,BS,lens,window,sinks,scale", [
    (14, 2, 64, 32, [600], -1, False, 0.125),
    (14, 2, 64, 16, SHORT, -1, False, 0.125),
    (15, 1, 64, 64, SHORT, 100, True, -0.125),
    (32, 8, 128, 32, SHORT, -1, True, 0.09),
    (32, 32, 128, 16, SHORT, 40, False, 0.09),    # many workgroups of four waves
    (64, 32, 64, 64, SHORT, -1, False, 0.0),
    (32, 8, 128, 16, LONG, -1, True, 0.09),       # the units of all dealt to runs
    (8, 2, 128, 64, LONG, 2100, False, -0.09),
    (16, 2, 64, 32, LONG, -1, False, 0.125),
])
def test_append_decode_is_store_and_attend(Hq, Hk, D, BS, lens, window, sinks, scale):
    q, k, v, kc, vc, pos, cs, slots, bt, sl = _inputs(Hq, Hk, D, BS, lens, D + BS)
    if len(lens) > 2:
        slots[1] = -1  # this one's token is in the cache
    sk = torch.linspace(-2, 2, Hq, device="cuda") if sinks else None
    kw = dict(sliding_window=window, sinks=sk, max_seq_len=max(lens))
    kc2, vc2, q2 = kc.clone(), vc.clone(), q.clone()
    ops.rope_and_cache(q2, k, v, kc2, vc2, pos, cs, slots)
    want = ops.paged_attention_decode(q2, kc2, vc2, bt, sl, scale, **kw)
    before = q.clone()
    out = ops.rope_cache_attention_decode(q, k, v, kc, vc, pos, cs, slots, bt, sl,
                                          scale, **kw)
    assert torch.equal(out, want)
    assert torch.equal(kc, kc2) and torch.equal(vc, vc2) and torch.equal(q, before)


@pytest.mark.parametrize("Hq,Hk,D,BS,lens", [
    (14, 2, 64, 16, SHORT), (32, 8, 128, 32, SHORT), (32, 32, 128, 64, SHORT),
    (32, 8, 128, 16, LONG), (16, 2, 64, 64, LONG),
])
def test_append_decode_over_stale_slots(Hq, Hk, D, BS, lens):
    """The token's own place and those behind it hold NaN before."""
    q, k, v, kc, vc, pos, cs, slots, bt, sl = _inputs(Hq, Hk, D, BS, lens, D + BS)
    for i, n in enumerate(lens):
        page, at = int(bt[i, (n - 1) // BS]), (n - 1) % BS
        if i == 1:
            slots[1], at = -1, at + 1  # this one's token is in the cache
        kc[page, :, at:] = float("nan")
        vc[page, :, :, at:] = float("nan")
    kc2, vc2, q2 = kc.clone(), vc.clone(), q.clone()
    ops.rope_and_cache(q2, k, v, kc2, vc2, pos, cs, slots)
    want = ops.paged_attention_decode(q2, kc2, vc2, bt, sl, 0.1, max_seq_len=max(lens))
    out = ops.rope_cache_attention_decode(q, k, v, kc, vc, pos, cs, slots, bt, sl, 0.1,
                                          max_seq_len=max(lens))
    assert out.isfinite().all() and torch.equal(out, want)
    assert torch.equal(kc.view(torch.int16), kc2.view(torch.int16))
    assert torch.equal(vc.view(torch.int16), vc2.view(torch.int16))


def test_append_decode_in_a_graph():
    """Lengths, places and values of each replay are those in memory then."""
    q, k, v, kc, vc, pos, cs, slots, bt, sl = _inputs(32, 8, 128, 32, [700, 40, 512], 5)
    args = (q, k, v, kc, vc, pos, cs, slots, bt, sl, 0.09)
    ops.rope_cache_attention_decode(*args, max_seq_len=1024)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.rope_cache_attention_decode(*args, max_seq_len=1024)
    for step in range(3):
        sl.sub_(1)
        pos.sub_(1)
        slots.copy_(bt.gather(1, ((sl - 1) // 32).long()[:, None])[:, 0] * 32
                    + (sl - 1) % 32)
        q.mul_(0.5)
        kc2, vc2, q2 = kc.clone(), vc.clone(), q.clone()
        ops.rope_and_cache(q2, k, v, kc2, vc2, pos, cs, slots)
        want = ops.paged_attention_decode(q2, kc2, vc2, bt, sl, 0.09, max_seq_len=1024)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(kc, kc2) and torch.equal(vc, vc2)


def test_append_decode_refuses_what_it_has_no_kernel_for():
    q, k, v, kc, vc, pos, cs, slots, bt, sl = _inputs(8, 2, 64, 32, [40, 70], 1)

    def call(**kw):
        a = dict(q=q, k=k, v=v, k_cache=kc, v_cache=vc, positions=pos, cos_sin=cs,
                 slot_mapping=slots, block_tables=bt, seq_lens=sl, scale=0.125,
                 max_seq_len=70)
        a.update(kw)
        return ops.rope_cache_attention_decode(**a)

    assert call() is not None
    assert call(cos_sin=cs[:, :32].contiguous()) is None      # part of a head turned
    assert call(k_cache=kc.to(torch.float8_e4m3fn),
                v_cache=vc.to(torch.float8_e4m3fn)) is None
    assert call(max_seq_len=None) is None
    assert call(q=q.float()) is None
    assert call(k=torch.cat([k, k], 2)[..., ::2]) is None     # values apart
    assert call(positions=pos[:1]) is None
    q16 = torch.cat([q] * 4, 1)  # 16 query heads leave the key no column
    assert call(q=q16) is None
