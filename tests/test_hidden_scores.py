"""The arithmetic of a tile in the attention kernels, in fp32 on the CPU: weights
are exp2(fma(score, c, -m)), m is the running maximum of rounded products score * c,
and what came before is multiplied by exp2(m_old - m_new)."""

import numpy as np
import pytest

F = np.float32


def _fma(a, b, c):
    """One rounding: the product of two fp32 values is exact in 64 bits."""
    return (a.astype(np.float64) * np.float64(b) + np.float64(c)).astype(F)


def _attend(tiles, seen, v, c, hidden, start):
    m, l, o = F(start), F(0), F(0)
    with np.errstate(all="ignore"):
        for s, on, x in zip(tiles, seen, v):
            s = np.where(on, s, F(hidden)).astype(F)
            mx = F(s.max() * F(c))
            if mx > m:
                f = np.exp2(F(m - mx))
                m, l, o = mx, F(l * f), F(o * f)
            p = np.exp2(_fma(s, F(c), -m))
            l = F(l + p.sum(dtype=F))
            o = F(o + (p * x).sum(dtype=F))
    return m, l, o


SCALES = [0.0, 1e-6, 1 / 128, 0.01, 0.0442, 1 / 12, 128 ** -0.5, 0.1, 0.125,
          80 ** -0.5, 192 ** -0.5, 0.25, 0.37, 0.6, 1.0, 3.0]


@pytest.mark.parametrize("hide", [(0,), (0, 1), (2,), (0, 2), ()])
def test_tiles_without_a_visible_key_leave_the_sums_alone(hide):
    rng = np.random.default_rng(len(hide))
    for scale in SCALES:
        c = max(F(scale) * F(1.44269504), F(1e-20))
        s = (rng.standard_normal((3, 64)) * 8).astype(F)
        v = rng.standard_normal((3, 64)).astype(F)
        seen = rng.random((3, 64)) < 0.5
        seen[:, 5] = True
        seen[list(hide)] = False
        m, l, o = _attend(s, seen, v, c, -np.inf, -1e30)
        w = np.exp(s[seen].astype(np.float64) * scale
                   - (s[seen].astype(np.float64) * scale).max())
        # 200 fp32 operations a sum, scores of up to 2^7 in the exponent
        assert abs(o / l - (w * v[seen]).sum() / w.sum()) < 1e-4, (scale, hide)


def test_a_split_that_sees_nothing_has_no_weight():
    s = np.ones((2, 64), F)
    for scale in SCALES:
        c = max(F(scale) * F(1.44269504), F(1e-20))
        m, l, o = _attend(s, np.zeros((2, 64), bool), s, c, -np.inf, -1e30)
        assert (m, l, o) == (F(-1e30), 0, 0)


def test_a_finite_hidden_score_is_rounded_once():
    """Why it is not finite: the weight's exponent is the product's rounding."""
    s = np.ones((1, 64), F)
    bad = [x for x in SCALES
           if not np.isfinite(_attend(s, np.zeros((1, 64), bool), s,
                                      F(x) * F(1.44269504), -1e30, -1e30)[1])]
    assert 0.125 in bad
