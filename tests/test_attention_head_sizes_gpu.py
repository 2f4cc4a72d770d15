"""GPU parity of 16-bit attention for head sizes other than 64 and 128: multiples of 8 on the matrix cores
(rows padded to 64 or 128 in LDS), the rest on the scalar kernel; block edges, masks, negative scale.

Bound, with P the exact probabilities: a score is off by at most (D + 2) 2^-24 of scale sum |q||k|, a probability
by twice the largest of those in relative terms, 2^-22 for its exponential and Skv 2^-24 for its sums; the
result is that times sum P |v|, rounded once to its type."""
import numpy as np
import pytest
import torch

from tests.util import NAME, as_f64, to_dev

pytestmark = pytest.mark.gpu
ROUNDOFF = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _reference(q, k, v, scale, causal, mask):
    s = (q @ np.swapaxes(k, -1, -2)) * scale
    err = (q.shape[-1] + 2) * 2.0 ** -24 * np.max((np.abs(q) @ np.swapaxes(np.abs(k), -1, -2)) * abs(scale))
    if mask is not None:
        s = s + mask
    if causal:
        s = np.where(np.arange(s.shape[-1]) > np.arange(s.shape[-2])[:, None], -np.inf, s)
    m = s.max(-1, keepdims=True)
    p = np.exp(s - np.where(np.isfinite(m), m, 0))
    p = p / np.maximum(p.sum(-1, keepdims=True), 1e-300)
    return p @ v, (2 * err + 2.0 ** -22 + (s.shape[-1] + 8) * 2.0 ** -24) * (p @ np.abs(v))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("D", [4, 8, 24, 32, 40, 56, 72, 80, 96, 104, 120, 136])
@pytest.mark.parametrize("B,H,Sq,Skv,causal,mask", [(1, 1, 1, 1, False, False), (2, 3, 33, 65, False, True), (1, 8, 127, 127, True, False), (2, 4, 130, 200, True, True),
                                                    (1, 2, 257, 63, True, False), (3, 1, 5, 321, False, False)], ids=lambda v: str(v))
def test_head_sizes(B, H, Sq, Skv, causal, mask, D, dtype):
    from metalhlo_amd import kernels
    rng = np.random.default_rng(D)
    q, k, v = (to_dev(rng.standard_normal((B, H, n, D)), dtype) for n in (Sq, Skv, Skv))
    md = None
    if mask:
        m = rng.standard_normal((B, 1, Sq, Skv))
        m[..., Skv // 2:] = -np.inf
        m[0, 0, Sq // 2] = -np.inf           # one row hides every key: zeros
        md = to_dev(m, dtype)
    scale = -0.3 if Skv == 65 else D ** -0.5
    guard = torch.full((B * H * Sq * D + 64,), float("nan"), dtype=dtype, device="cuda")
    got = kernels.flash_attention(q, k, v, scale=scale, is_causal=causal, mask=md, out=guard[:-64].view(B, H, Sq, D))
    e, bound = _reference(as_f64(q), as_f64(k), as_f64(v), scale, causal, None if md is None else as_f64(md))
    diff = np.abs(as_f64(got) - e)
    tiny = 2.0 ** -24 if dtype == torch.float16 else 0.0       # f16's smallest numbers are evenly spaced
    assert np.all(diff <= bound + ROUNDOFF[dtype] * (np.abs(e) + bound) + tiny), (diff.max(), np.abs(e).max())
    assert torch.isnan(guard[-64:]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("D", [24, 40, 80, 96, 120])
@pytest.mark.parametrize("causal,mask", [(True, False), (False, False), (True, True)], ids=lambda v: str(v))
def test_values_that_are_not_finite(causal, mask, D, dtype):
    """An infinity or a NaN in V reaches the rows that see its key, as itself, and no other: rows in front of a causally
    hidden key (same 64-key block included) are those of clean operands, other columns and heads too."""
    from metalhlo_amd import kernels
    B, H, S = 2, 3, 200
    rng = np.random.default_rng(D)
    q, k, v = (to_dev(rng.standard_normal((B, H, S, D)) * 0.5, dtype) for _ in range(3))
    md = to_dev(rng.standard_normal((B, 1, S, S)), dtype) if mask else None
    e, bound = _reference(as_f64(q), as_f64(k), as_f64(v), D ** -0.5, causal, None if md is None else as_f64(md))
    plus, minus, nan = 131, 150, 190                       # keys
    w = v.clone()
    w[0, 1, plus, 3] = float("inf")
    w[0, 1, minus, D - 1] = float("-inf")
    w[1, 2, nan] = float("nan")
    got = as_f64(kernels.flash_attention(q, k, w, is_causal=causal, mask=md))
    sees = lambda key: np.arange(S) >= key if causal else np.ones(S, bool)  # noqa: E731
    want = e.copy()
    want[0, 1, sees(plus), 3] = np.inf
    want[0, 1, sees(minus), D - 1] = -np.inf
    want[1, 2, sees(nan)] = np.nan
    clean = np.isfinite(want)
    tiny = 2.0 ** -24 if dtype == torch.float16 else 0.0
    assert np.all(np.abs(got - e)[clean] <= (bound + ROUNDOFF[dtype] * (np.abs(e) + bound) + tiny)[clean])
    assert np.array_equal(got[~clean], want[~clean], equal_nan=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("D", [40, 96])
def test_probabilities_keep_their_fp32_bits(D, dtype):
    """Values of +1 and -1 under weights that differ by 2^-15 of themselves: what is left of their sum shows every bit
    a weight lost on its way into the product.  A score of -t (t below 1) is off by 2^-24, its exponential by 2^-22 in
    all and the sums of 130 keys by 2^-21 of the sum of weights."""
    from metalhlo_amd import kernels
    S, n = 130, 64
    q, k, v = (np.zeros((1, 2, S, D)) for _ in range(3))
    q[..., 0] = 0.5 + np.arange(S) / 512
    q[..., 1] = 2.0 ** -7
    k[..., 1:1 + n, 0] = k[..., 1 + n:1 + 2 * n, 0] = -1.0
    k[..., 1 + n:1 + 2 * n, 1] = 2.0 ** -8
    v[..., 1:1 + n, :], v[..., 1 + n:1 + 2 * n, :] = -1.0, 1.0
    q, k, v = (to_dev(x, dtype) for x in (q, k, v))
    got = as_f64(kernels.flash_attention(q, k, v, scale=1.0))
    e, _ = _reference(as_f64(q), as_f64(k), as_f64(v), 1.0, False, None)
    assert e.min() > 2.0 ** -17
    assert np.all(np.abs(got - e) <= 2.0 ** -21 + ROUNDOFF[dtype] * e)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
def test_small_probabilities_count(dtype):
    """A key of weight one whose value is zero, and weights of e^-21 on large values, far below f16's smallest number."""
    from metalhlo_amd import kernels
    S, D = 100, 72
    q, k, v = (np.zeros((1, 1, S, D)) for _ in range(3))
    q[..., :2] = 1.0
    k[..., 1:, 0], k[..., 1:, 1] = -20.0, -1.0
    v[..., 1:, :] = 60000.0
    q, k, v = (to_dev(x, dtype) for x in (q, k, v))
    got = as_f64(kernels.flash_attention(q, k, v, scale=1.0))
    e = 99 * np.exp(-21.0) * as_f64(v)[0, 0, 1, 0] / (1 + 99 * np.exp(-21.0))
    # (an exponent of 21 is off by 2^-19; f16's subnormal numbers do not come into it: e is 4.5e-3)
    assert np.all(np.abs(got - e) <= (2.0 ** -18 + ROUNDOFF[dtype]) * e)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("D,S,causal,unit", [(24, 70, False, 14), (96, 200, True, 14), (40, 130, True, 12), (72, 300, False, 13)], ids=lambda v: str(v))
def test_large_scores(D, S, causal, unit, dtype):
    """Scores of 2^24 to 2^38 that fp32 holds exactly (small integers times a power of two): the largest share the row."""
    from metalhlo_amd import kernels
    rng = np.random.default_rng(S)
    q, k = (to_dev(rng.integers(-3, 4, (1, 2, S, D)) * 2.0 ** unit, dtype) for _ in range(2))
    k[..., 1::3, :] = k[..., 0:1, :]                        # many equal keys
    v = to_dev(rng.standard_normal((1, 2, S, D)), dtype)
    got = as_f64(kernels.flash_attention(q, k, v, scale=1.0, is_causal=causal))
    s = as_f64(q) @ np.swapaxes(as_f64(k), -1, -2)
    if causal:
        s = np.where(np.arange(S) > np.arange(S)[:, None], -np.inf, s)
    p = (s == s.max(-1, keepdims=True)).astype(float)
    p /= p.sum(-1, keepdims=True)
    e, sums = p @ as_f64(v), (S + 8) * 2.0 ** -24 * (p @ np.abs(as_f64(v)))
    assert np.all(np.abs(got - e) <= sums + ROUNDOFF[dtype] * (np.abs(e) + sums) + 2.0 ** -24)
