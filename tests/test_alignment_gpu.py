"""Caches, activations and expert weights that begin at an odd place in memory."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from parallax_amd import ops


def _odd(t):
    """The same values, one element behind a multiple of 16 bytes."""
    flat = torch.empty(t.numel() + 16, dtype=t.dtype, device=t.device)[1 : t.numel() + 1]
    return flat.copy_(t.reshape(-1)).view(t.shape)


@pytest.mark.parametrize("fp8", [False, True])
def test_paged_caches(fp8):
    g = torch.Generator(device="cuda").manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    kc, vc, q = r(9, 2, 32, 64), r(9, 2, 64, 32), r(3, 8, 64)
    if fp8:
        kc, vc = (t.to(torch.float8_e4m3fn) for t in (kc, vc))
    bt = torch.arange(9, dtype=torch.int32, device="cuda").view(3, 3)
    sl = torch.tensor([70, 96, 5], dtype=torch.int32, device="cuda")
    for longest in (96, 5000):
        a, b = (ops.paged_attention_decode(q, k, v, bt, sl, 0.125, max_seq_len=longest)
                for k, v in ((kc, vc), (_odd(kc), _odd(vc))))
        assert torch.equal(a, b)
    ql = torch.tensor([1, 1, 1], dtype=torch.int32, device="cuda")
    a, b = (ops.prefill_attention(q, k, v, bt, sl, ql, 0.125)
            for k, v in ((kc, vc), (_odd(kc), _odd(vc))))
    assert torch.equal(a, b)


@pytest.mark.parametrize("fp8", [False, True])
def test_latent_cache(fp8):
    g = torch.Generator(device="cuda").manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    cache, ql, qp = r(9, 32, 576), r(3, 16, 512), r(3, 16, 64)
    if fp8:
        cache = cache.to(torch.float8_e4m3fn)
    bt = torch.arange(9, dtype=torch.int32, device="cuda").view(3, 3)
    sl = torch.tensor([70, 96, 5], dtype=torch.int32, device="cuda")
    a, b = (ops.mla_paged_attention_decode(ql, qp, c, bt, sl, 0.07)
            for c in (cache, _odd(cache)))
    assert torch.equal(a, b)


@pytest.mark.parametrize("fp8", [False, True])
def test_experts(fp8):
    g = torch.Generator(device="cuda").manual_seed(2)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, gu, dn = r(40, 128).bfloat16(), r(4, 128, 128) * 0.1, r(4, 128, 64) * 0.1
    ids = torch.randint(0, 4, (40, 2), generator=g, device="cuda")
    w = torch.rand(40, 2, generator=g, device="cuda")
    if fp8:
        (gu, gs), (dn, ds) = ops.quantize_fp8_weight(gu), ops.quantize_fp8_weight(dn)
        run = lambda x, u, d: ops.fused_moe_forward_fp8(x, u, gs, d, ds, ids, w)
    else:
        gu, dn = gu.bfloat16(), dn.bfloat16()
        run = lambda x, u, d: ops.fused_moe_forward(x, u, d, ids, w)
    assert torch.equal(run(x, gu, dn), run(_odd(x), _odd(gu), _odd(dn)))
