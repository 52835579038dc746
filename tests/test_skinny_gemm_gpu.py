"""Few rows against a large weight, its fp8 form and MLA's per-head products,
against fp32."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from parallax_amd import ops


def _rand(g, *s):
    return torch.randn(*s, generator=g, device="cuda")


@pytest.mark.parametrize("M,N,K", [
    (M, N, K) for M in (1, 8, 9, 16, 17, 32) for N, K in (
        (4, 64),        # one column of 128 bytes: waves without one
        (900, 896),     # a tile cut by the last row
        (4804, 2176),   # 32 rows a tile, deep rings
        (9604, 320),    # 64 rows a tile
    )
] + [
    (1, 2044, 2048), (5, 900, 4864), (8, 12, 2112),      # 8 rows a tile
    (33, 576, 2112), (64, 100, 2048), (64, 5000, 3072),  # K shared, odd parts
    (20, 1536, 7168), (32, 24576, 1408),                 # the same, fewer rows
    (65, 4100, 4096), (96, 28672, 320), (128, 36864, 256),  # 3 to 5 waves
    (127, 8192, 2112),
])
def test_linear_few_rows(M, N, K):
    """fp32 sums of exact products: 2^-8 of the result for its rounding, and
    K 2^-24 of the sum of magnitudes (< K here) for the sums."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = _rand(g, M, 2 * K).bfloat16()[:, K:]
    w = _rand(g, N, K).bfloat16()
    b = _rand(g, N).bfloat16()
    ext = ops._require_ext("skinny_gemm")
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    none = x.new_empty(0)
    assert ext.skinny_gemm(out, x, w, none, none, none, False)
    want = x.float() @ w.float().t()
    tol = dict(rtol=2 ** -8, atol=K * K * 2 ** -24)
    torch.testing.assert_close(out.float(), want, **tol)
    torch.testing.assert_close(ops.linear(x, w, b).float(), want + b.float(), **tol)


@pytest.mark.parametrize("M,N,K", [(1, 2044, 2048), (8, 12, 2112), (5, 4804, 2176),
                                   (40, 1536, 7168)])
def test_linear_infinities(M, N, K):
    """An infinite weight reaches its own column, an infinite value its own row."""
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w = _rand(g, M, K).bfloat16(), _rand(g, N, K).bfloat16()
    want = ops.linear(x, w)
    w[3, K - 1] = w[N - 1, 0] = float("inf")
    x[M - 1, K // 2] = float("inf")
    got = ops.linear(x, w)
    assert not got[:, [3, N - 1]].isfinite().any() and not got[M - 1].isfinite().any()
    got[:, [3, N - 1]] = want[:, [3, N - 1]]
    assert torch.equal(got[:M - 1], want[:M - 1])


def test_linear_without_a_kernel():
    """Odd widths and misaligned rows take the library and agree."""
    g = torch.Generator(device="cuda").manual_seed(0)
    for M, N, K in ((5, 8, 72), (3, 6, 64), (33, 64, 64), (96, 576, 7168),
                    (129, 4096, 512)):
        x, w = _rand(g, M, K).bfloat16(), _rand(g, N, K).bfloat16()
        torch.testing.assert_close(
            ops.linear(x, w).float(), x.float() @ w.float().t(), rtol=2 ** -8,
            atol=K * K * 2 ** -24)
    x = _rand(g, 4, 65).bfloat16()[:, 1:]
    w = _rand(g, 64, 64).bfloat16()
    torch.testing.assert_close(
        ops.linear(x, w).float(), x.float() @ w.float().t(), rtol=2 ** -8, atol=1e-3)


def test_linear_of_rows_far_apart():
    """Rows whose places do not fit 32 bits (the last token of every long prompt,
    say)."""
    g = torch.Generator(device="cuda").manual_seed(7)
    apart = 24 << 20
    buf = torch.empty(100 * apart, dtype=torch.bfloat16, device="cuda")
    for M in (100, 100, 24):
        x = buf.as_strided((M, 512), (apart * (100 // M), 1))
        x.copy_(_rand(g, M, 512))
        w = _rand(g, 28672, 512).bfloat16()
        torch.testing.assert_close(
            ops.linear(x, w).float(), x.float() @ w.float().t(), rtol=2 ** -8,
            atol=512 ** 2 * 2 ** -24)
    lat = buf.as_strided((34, 2, 512), (apart * 2, 512, 1))
    lat.copy_(_rand(g, 34, 2, 512))
    uv = _rand(g, 2, 128, 512).bfloat16()
    torch.testing.assert_close(
        ops.mla_project_out(lat, uv).float(),
        torch.einsum("bhr,hvr->bhv", lat.float(), uv.float()), rtol=2 ** -8,
        atol=512 ** 2 * 2 ** -24)


@pytest.mark.parametrize("M,N,K,own", [
    (6, 40964, 64, True), (7, 40964, 64, False), (16, 40964, 64, False),
    (17, 40964, 64, True), (16, 40960, 64, True), (16, 40964, 2048, True),
    (33, 40964, 64, False), (100, 40964, 2048, True),
    (33, 5120, 2560, False), (64, 8192, 2048, True), (65, 8192, 2048, False),
    (65, 4096, 3584, True), (40, 256, 7168, True), (40, 256, 4096, False),
])
def test_linear_takes_the_faster_side(M, N, K, own):
    """Both sides of the lines between the kernels and the library agree."""
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w = _rand(g, M, K).bfloat16(), _rand(g, N, K).bfloat16()
    ext = ops._require_ext("few_rows")
    none = x.new_empty(0)
    got = ext.few_rows(x, w, none, none, none, False)
    assert (got is not None) == own
    torch.testing.assert_close(
        ops.linear(x, w).float(), x.float() @ w.float().t(), rtol=2 ** -8,
        atol=K * K * 2 ** -24)


def test_linear_gradients():
    """Rows apart and odd widths, which torch's product takes, have gradients."""
    g = torch.Generator(device="cuda").manual_seed(3)
    for M, N, K, cut in ((6, 64, 128, True), (6, 68, 128, False)):
        base = _rand(g, M, 2 * K if cut else K).bfloat16().requires_grad_()
        w = _rand(g, N, K).bfloat16().requires_grad_()
        b = _rand(g, N).bfloat16().requires_grad_()
        y = ops.linear(base[:, :K], w, b)
        y.float().sum().backward()
        torch.testing.assert_close(b.grad.float(), torch.full((N,), float(M), device="cuda"))
        torch.testing.assert_close(
            base.grad[:, :K].float(),
            w.detach().float().sum(0).expand(M, K), rtol=2 ** -7, atol=2 ** -7)
        torch.testing.assert_close(
            w.grad.float(), base.detach()[:, :K].float().sum(0).expand(N, K),
            rtol=2 ** -7, atol=2 ** -7)
        with torch.no_grad():
            torch.testing.assert_close(ops.linear(base[:, :K], w, b).float(), y.float(),
                                       rtol=2 ** -7, atol=2 ** -7)


def test_linear_allocates_its_result_once():
    """Also where no kernel for few rows takes the product."""
    g = torch.Generator(device="cuda").manual_seed(4)
    for M, N, K in ((96, 576, 7168), (33, 64, 64), (8, 900, 896)):
        x, w = _rand(g, M, K).bfloat16(), _rand(g, N, K).bfloat16()
        ops.linear(x, w)
        n = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
        before = n()
        y = ops.linear(x, w)
        assert n() - before == 1 and y.shape == (M, N)


def test_linear_of_no_columns():
    """Refused by the kernels, whose deals of columns assume one."""
    ext = ops._require_ext("skinny_gemm")
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")
    for M, N, K in ((4, 64, 0), (40, 64, 0), (4, 0, 64)):
        assert not ext.skinny_gemm(z(M, N), z(M, K), z(N, K), z(0), z(0), z(0), False)


@pytest.mark.parametrize("M,N,K", [(1, 64, 128), (7, 4800, 5120), (16, 64, 256),
                                   (30, 9600, 384), (40, 256, 512),
                                   (12, 36864, 256), (50, 1000, 4224),
                                   (96, 36864, 512), (128, 8192, 4096)])
def test_linear_fp8_rows(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M)
    x = _rand(g, M, K).bfloat16()
    w = _rand(g, N, K).to(torch.float8_e4m3fn)
    ws = torch.tensor([0.37], device="cuda")
    xs = (x.float().abs().amax() / 448.0).clamp_min(1e-8).reshape(1)
    xq = (x.float() / xs).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    want = (xq.float() @ w.float().t()) * (xs * ws)
    torch.testing.assert_close(
        ops.linear_fp8(x, w, ws).float(), want, rtol=2 ** -8,
        atol=K * K * 2 ** -24)


@pytest.mark.parametrize("M,N,K,kind,own", [(M, *c) for M in (33, 64, 65, 97, 128) for c in (
    (8, 64, "bias", True), (1152, 896, "bias", True), (1288, 4928, "", True),  # 16 rows
    (2056, 960, "bias", True), (2904, 2112, "", True), (4104, 64, "gated", None),  # 32
    (2184, 5952, "", True),
    (9680, 64, "gated", None), (7664, 896, "gated", True),                     # 64
    (904, 2176, "fp8", True), (2568, 3968, "fp8", True), (7664, 1024, "fp8gated", None),
    (13008, 1024, "", False), (240, 2112, "", False),
    (1156, 896, "", False), (1152, 896, "apart", False),  # torch's product as before
)] + [(M, *c) for M in (129, 300, 384) for c in (
    (8, 64, "bias", True), (904, 896, "bias", True), (640, 1024, "gated", True),
    (904, 2176, "fp8", True), (3080, 2048, "", False), (904, 896, "apart", False),
)] + [(385, 896, 896, "", False)])
def test_linear_in_pieces_of_32_rows(M, N, K, kind, own):
    """Cut tiles and pieces, against fp32. Infinities stay in their rows and columns.
    own: whether a kernel takes it, whatever M is."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    fp8, gated = kind.startswith("fp8"), kind.endswith("gated")
    x, w = _rand(g, M, K).bfloat16(), _rand(g, N, K).bfloat16()
    if kind == "apart":
        x = torch.cat([x, x], 1)[:, :K]
    none, one = x.new_empty(0), torch.ones(1, device="cuda")
    b = _rand(g, N).bfloat16() if kind == "bias" else none
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
    run = lambda: ops._require_ext("few_rows").few_rows(
        x, w, b, one if fp8 else none, one if fp8 else none, gated)
    got = run()
    assert own is None or (got is not None) == own
    if got is None:
        return
    want = x.float() @ w.float().t()
    if b.numel():
        want += b.float()
    atol = K * K * 2 ** -24
    if gated:   # both products rounded to bf16, |silu'| < 1.1, the result rounded
        a, u = want.bfloat16().float().chunk(2, dim=1)
        s = torch.nn.functional.silu(a)
        want = s * u
        atol = (atol + 2 ** -7 * a.abs()) * 1.1 * u.abs() + (
            atol + 2 ** -7 * u.abs()) * s.abs() + 1e-6
    assert ((got.float() - want).abs() <= atol + 2 ** -7 * want.abs()).all()
    if fp8 or gated:
        return
    w[N - 1, 0] = x[M - 1, K - 1] = float("inf")
    again = run()
    assert not again[M - 1].isfinite().any() and not again[:, N - 1].isfinite().any()
    assert torch.equal(again[:-1, :-1], got[:-1, :-1])


@pytest.mark.parametrize("M,N,K,kind,own", [
    (128, 5056, 640, "", False), (128, 5056, 640, "bias", True),      # 64 rows a tile
    (40, 9344, 512, "", False), (40, 9344, 512, "gated", True),
    (192, 5184, 768, "", False), (256, 2240, 896, "", False),
    (96, 7296, 512, "fp8", False), (80, 8640, 1792, "fp8", False),
    (160, 4096, 960, "gated", True), (161, 4096, 960, "gated", False),
    (97, 2880, 2560, "fp8", False), (97, 2560, 2560, "fp8", True),    # 32
    (128, 2584, 1472, "", False), (128, 2560, 1472, "", True),
    (128, 2584, 1472, "bias", True), (129, 2432, 1472, "", True), (128, 3072, 1536, "", True), (128, 3080, 1536, "", False),
])
def test_pieces_leave_the_library_what_it_does_faster(M, N, K, kind, own):
    """Wide tiles that save no launch, and short rows in more blocks than the chip takes at
    once, are the library's; both sides of these lines agree with fp32."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    fp8, gated = kind == "fp8", kind == "gated"
    x, w = _rand(g, M, K).bfloat16(), _rand(g, N, K).bfloat16()
    none, one = x.new_empty(0), torch.ones(1, device="cuda")
    b = _rand(g, N).bfloat16() if kind == "bias" else None
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
    got = ops._require_ext("few_rows").few_rows(
        x, w, none if b is None else b, one if fp8 else none, one if fp8 else none, gated)
    assert (got is not None) == own
    y = (ops.linear_fp8_quantized(x, one, w, one) if fp8 else
         ops.linear_silu_and_mul(x, w) if gated else ops.linear(x, w, b)).float()
    want = x.float() @ w.float().t()
    if b is not None:
        want += b.float()
    # the library's bias comes behind a rounding of its own
    atol = K * K * 2 ** -24 + (0 if b is None else 2 ** -8 * (want - b.float()).abs())
    if gated:   # both products rounded to bf16, |silu'| < 1.1, the result rounded
        a, u = want.bfloat16().float().chunk(2, dim=1)
        s = torch.nn.functional.silu(a)
        want = s * u
        atol = (atol + 2 ** -7 * a.abs()) * 1.1 * u.abs() + (
            atol + 2 ** -7 * u.abs()) * s.abs() + 1e-6
    assert ((y - want).abs() <= atol + 2 ** -7 * want.abs()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 7, 2048, 2057, 700001])
def test_quantize_fp8_tensor(dtype, n):
    """Bytes and scale as the torch operations give them, also with zeros,
    infinities and NaN."""
    g = torch.Generator(device="cuda").manual_seed(n)
    ext = ops._require_ext("quantize_fp8_tensor")
    base = (_rand(g, n + 1) * 100).to(dtype)
    for x in (base[1:].clone(), base[1:], torch.zeros_like(base[1:])):
        for special in (None, float("inf"), float("nan")):
            x = x.clone() if special is not None else x
            if special is not None:
                x[n // 2] = special
            q, s = ext.quantize_fp8_tensor(x)
            xf = x.float()
            want_s = (xf.abs().amax() / 448.0).clamp_min(1e-8).reshape(1)
            want = (xf / want_s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
            assert torch.equal(s.view(torch.int32), want_s.view(torch.int32)) or (
                s.isnan().item() and want_s.isnan().item())
            a, b = q.float(), want.float()
            assert torch.equal(a.isnan(), b.isnan())
            assert torch.equal(a.nan_to_num(), b.nan_to_num())


# both passes' grids at and past their ends: 1,024 and 2,048 workgroups of 2,048 values
@pytest.mark.parametrize("n", [1024 * 2048, 1024 * 2048 + 1, 2048 * 2048 + 1, 9000003])
@pytest.mark.parametrize("at", [0, -1])
def test_quantize_fp8_tensor_large(n, at):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = _rand(g, n).bfloat16()
    x[at] = 1000.0
    q, s = ops._require_ext("quantize_fp8_tensor").quantize_fp8_tensor(x)
    want_s = (x.float().abs().amax() / 448.0).reshape(1)
    want = (x.float() / want_s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    assert torch.equal(s, want_s)
    assert torch.equal(q.view(torch.uint8), want.view(torch.uint8))


@pytest.mark.parametrize("B,H", [(1, 16), (8, 3), (16, 128), (33, 16), (70, 2)])
def test_mla_products(B, H):
    g = torch.Generator(device="cuda").manual_seed(B)
    q = _rand(g, B, H, 192).bfloat16()[..., :128]
    uk, uv = (_rand(g, H, 128, 512).bfloat16() for _ in range(2))
    lat = _rand(g, B, H, 512).bfloat16()
    torch.testing.assert_close(
        ops.mla_absorb(q, uk).float(),
        torch.einsum("bhd,hdr->bhr", q.float(), uk.float()), rtol=2 ** -8,
        atol=128 ** 2 * 2 ** -24)
    torch.testing.assert_close(
        ops.mla_project_out(lat, uv).float(),
        torch.einsum("bhr,hvr->bhv", lat.float(), uv.float()), rtol=2 ** -8,
        atol=512 ** 2 * 2 ** -24)
    # other widths: the torch products
    torch.testing.assert_close(
        ops.mla_absorb(q[..., :96], uk[:, :96]).float(),
        torch.einsum("bhd,hdr->bhr", q[..., :96].float(), uk[:, :96].float()),
        rtol=2 ** -8, atol=1e-2)


def test_mla_products_of_weights_in_other_orders():
    """Views of a fused weight, rows apart or transposed, and a batch of none."""
    g = torch.Generator(device="cuda").manual_seed(1)
    q = _rand(g, 5, 3, 128).bfloat16()
    lat = _rand(g, 5, 3, 512).bfloat16()
    fused = _rand(g, 3, 256, 512).bfloat16()
    turned = _rand(g, 3, 512, 128).bfloat16().transpose(1, 2)
    for w in (fused[:, :128], fused[:, 128:], turned):
        torch.testing.assert_close(
            ops.mla_absorb(q, w).float(),
            torch.einsum("bhd,hdr->bhr", q.float(), w.float()), rtol=2 ** -8,
            atol=128 ** 2 * 2 ** -24)
        torch.testing.assert_close(
            ops.mla_project_out(lat, w).float(),
            torch.einsum("bhr,hvr->bhv", lat.float(), w.float()), rtol=2 ** -8,
            atol=512 ** 2 * 2 ** -24)
    assert ops.mla_absorb(q[:, :0], fused[:0, :128]).shape == (5, 0, 512)
    assert ops.mla_project_out(lat[:0], fused[:, :128]).shape == (0, 3, 128)


@pytest.mark.parametrize("M,I,K", [
    (1, 8, 128), (8, 456, 896), (9, 2408, 2176), (16, 4872, 384), (32, 4872, 384),
    (20, 768, 11264), (33, 304, 4224), (64, 2408, 4224), (96, 14336, 256),
    (128, 18432, 256), (3, 104, 72), (130, 64, 256),
])
def test_linear_silu_and_mul(M, I, K):
    """Gate and up are rounded to bf16 (2^-8 of each at most), their function and the
    result's rounding follow; |silu'| < 1.1."""
    g = torch.Generator(device="cuda").manual_seed(M + I)
    x = _rand(g, M, K).bfloat16()
    w = (_rand(g, 2 * I, K) * K ** -0.5).bfloat16()
    b = _rand(g, 2 * I).bfloat16()
    out = ops.linear_silu_and_mul(x, w, b)
    y = x.float() @ w.float().t() + b.float()
    gate, up = y[:, :I], y[:, I:]
    silu = torch.nn.functional.silu(gate)
    want = silu * up
    # where the library has the product, it is rounded before the bias as well:
    # gate and up are off by 2^-8 of themselves and of what they were without it
    p = y - b.float()
    e = (y.abs() + p.abs()) * 2 ** -8
    bound = (1.1 * e[:, :I] * up.abs() + silu.abs() * e[:, I:]
             + want.abs() * 2 ** -8 + 1e-3)
    assert ((out.float() - want).abs() <= bound).all()
