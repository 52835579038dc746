"""hipBLASLt fp8 products: every pick of the tuner applies both scales."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from parallax_amd import ops


@pytest.mark.parametrize("M,N,K", [(40, 256, 512), (48, 576, 1024), (100, 512, 7168),
                                   (300, 256, 512)])
def test_fp8_scales(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.float8_e4m3fn)
    w = torch.randn(N, K, generator=g, device="cuda").to(torch.float8_e4m3fn)
    xs, ws = torch.tensor([0.011], device="cuda"), torch.tensor([0.37], device="cuda")
    y = ops._require_ext("lt_linear_fp8").lt_linear_fp8(x, w, xs, ws)
    want = (x.float() @ w.float().t()) * (xs * ws)
    # bf16 results, fp32 sums of K products below 100 * scales
    torch.testing.assert_close(y.float(), want, rtol=2 ** -8, atol=1e-3)
