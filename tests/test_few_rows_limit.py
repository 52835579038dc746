"""Which products ops.linear() hands to the kernels for few rows, by its limits alone."""

import types

import pytest
import torch

from parallax_amd import ops


@pytest.mark.parametrize("limit,tried", [
    (0, []), (1, [1]), (16, [1, 16]), (127, [1, 16, 17, 48, 127]),
    (128, [1, 16, 17, 48, 127, 128, 129, 384]),
    (200, [1, 16, 17, 48, 127, 128, 129, 384]),
])
def test_no_more_rows_than_the_limit_says(limit, tried, monkeypatch):
    """Below 128 the limit is that of all kernels, from there on small weights have some
    up to 384 rows; 0 leaves every product to the library."""
    asked = []
    monkeypatch.setattr(ops, "SKINNY_GEMM_MAX_M", limit)
    monkeypatch.setattr(ops, "_require_ext", lambda name: types.SimpleNamespace(
        few_rows=lambda x, *a: asked.append(x.shape[0])))
    w = torch.empty(896, 896, dtype=torch.bfloat16)
    for rows in (1, 16, 17, 48, 127, 128, 129, 384, 385):
        ops._few_rows(torch.empty(rows, 896, dtype=torch.bfloat16), w)
    assert asked == tried


def test_large_weights_have_128_rows_at_most(monkeypatch):
    asked = []
    monkeypatch.setattr(ops, "_require_ext", lambda name: types.SimpleNamespace(
        few_rows=lambda x, *a: asked.append(x.shape[0])))
    w = torch.empty(ops.PIECES_MAX_BYTES // 128 + 1, 64, dtype=torch.bfloat16)
    for rows in (128, 129):
        ops._few_rows(torch.empty(rows, 64, dtype=torch.bfloat16), w)
    assert asked == [128]


@pytest.mark.skipif(not ops.has_extension(), reason="the extension is not built")
def test_the_limits_are_the_kernels_own():
    limits = ops._require_ext("skinny_pieces_limits").skinny_pieces_limits()
    assert limits == (ops.PIECES_MAX_M, ops.PIECES_MAX_BYTES)
