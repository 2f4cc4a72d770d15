"""GPU parity of the row kernels at the places where rows of any length and alignment can go wrong: heads and
tails of every size, the borders between the numbers of threads and vectors per thread, tensors that start
inside a 16-byte line."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.util import NAME, TOL, as_f64, assert_close, to_dev

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16, torch.float16]
COLS = [1, 7, 9, 511, 513, 1023, 1025, 2047, 2051, 4099, 8191, 8193, 8200, 16390, 32771, 65537]


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: NAME[d])
@pytest.mark.parametrize("cols", COLS)
def test_rows_of_any_length(cols, dtype):
    from metalhlo_amd import kernels
    rng = np.random.default_rng(cols)
    for start in (0, 1, 3):                       # elements in front of the tensor
        x = to_dev(rng.standard_normal(5 * cols + start) * 2 + 0.5, dtype)[start:].view(5, cols)
        g, b = (to_dev(rng.standard_normal(cols) * 0.1 + c, dtype) for c in (1.0, 0.0))
        x64 = as_f64(x)
        # softmax: e^x of 16-bit rows sums to 1 within the types' rounding; the others as the operator tests do
        assert_close(kernels.softmax(x), oracle.softmax(x64), TOL[dtype], f"softmax {cols}+{start}")
        assert_close(kernels.layer_norm(x, g, b), oracle.layer_norm(x64, as_f64(g), as_f64(b), 1e-5), TOL[dtype], f"layer_norm {cols}+{start}")
        assert_close(kernels.rms_norm(x, g), oracle.rms_norm(x64, as_f64(g), 1e-5), TOL[dtype], f"rms_norm {cols}+{start}")
        assert_close(kernels.bias_gelu(x, b), oracle.bias_gelu(x64, as_f64(b)), TOL[dtype], f"bias_gelu {cols}+{start}")


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: NAME[d])
@pytest.mark.parametrize("cols", COLS)
def test_argmax_of_any_length(cols, dtype):
    """Ties take the lowest index, a NaN wins over any number and the first NaN over later ones."""
    from metalhlo_amd import kernels
    rng = np.random.default_rng(cols)
    x = np.round(rng.standard_normal((6, cols)) * 2)                    # many ties
    x[1] = -np.inf
    x[2, :] = 5.0
    x[3, cols // 2:] = np.nan
    for start in (0, 1):
        t = to_dev(np.concatenate([np.zeros(start), x.reshape(-1)]), dtype)[start:].view(6, cols)
        idx, val = kernels.argmax(t, torch.int64, return_values=True)
        e = np.array([np.flatnonzero(np.isnan(r))[0] if np.isnan(r).any() else int(np.argmax(r)) for r in x])
        assert np.array_equal(idx.cpu().numpy(), e)
        assert np.array_equal(as_f64(val), as_f64(t)[np.arange(6), e], equal_nan=True)


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: NAME[d])
@pytest.mark.parametrize("cols", [3, 64, 513, 768, 1025, 3072, 4096, 8200, 16391, 50257, 140001])
def test_softmax_at_the_ends_of_the_type(cols, dtype):
    """Rows of large numbers up to the ends of the type, where a maximum times log2(e) is rounded by more than a weight
    can stand and in the end leaves fp32: equal elements share the row, an element one representable step below has
    the weight of its distance.  One column count per row kernel and number of threads.  An exponent of x is off by
    2^-24 |x| (|x| below 150 where the weight is not zero), the sum of n weights by n 2^-24; one rounding follows."""
    from metalhlo_amd import kernels
    low, high = float(torch.finfo(dtype).min), float(torch.finfo(dtype).max)
    ulp = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    rows = []
    for m in [low, low * 0.75, low * 0.5, high * 0.5, high * 0.75, high] + [s * 2.0 ** e for e in (13, 14, 15, 16, 17, 24, 31, 40, 100, 126, 127) for s in (-1.0, 1.25) if 2.0 ** e * 1.25 < high]:
        r = np.full(cols, m)
        rows.append(r.copy())                                   # equal elements: 1 / n
        r[1::3] = max(low, m - 2 * ulp * abs(m))
        rows.append(r.copy())
        r[0::3] = low
        rows.append(r.copy())
        r[cols // 2] = -np.inf
        rows.append(r)
    r = np.full(cols, -np.inf)
    r[cols - 1] = low                                           # one element of weight 1
    rows.append(r)
    x = to_dev(np.stack(rows), dtype)
    x64 = as_f64(x)
    e = np.exp(x64 - x64.max(-1, keepdims=True))
    e /= e.sum(-1, keepdims=True)
    tiny = 2.0 ** -24 if dtype == torch.float16 else 2.0 ** -126    # the smallest normal fp32 number, f16's even spacing
    for start in (0, 1):                                        # elements in front of the tensor
        t = torch.cat([x.new_zeros(start), x.reshape(-1)])[start:].view(x.shape)
        got = as_f64(kernels.softmax(t))
        bad = ~(np.abs(got - e) <= ((cols + 300) * 2.0 ** -24 + ulp) * e + tiny)
        assert not bad.any(), (start, x64[bad][:4], got[bad][:4], e[bad][:4])


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: NAME[d])
@pytest.mark.parametrize("cols", [3, 7, 513, 1025, 3001, 16391, 50257])
def test_layer_norm_of_equal_elements(cols, dtype):
    """Rows of one large value: its multiples are exact in fp32, so the mean is the value, the variance zero and the result beta."""
    from metalhlo_amd import kernels
    beta = to_dev(np.random.default_rng(cols).standard_normal(cols), dtype)
    x = torch.tensor([12288.0, -49152.0, 1.5], dtype=dtype, device="cuda").repeat_interleave(cols).view(3, cols)
    got = kernels.layer_norm(x, torch.full((cols,), 2.0, dtype=dtype, device="cuda"), beta)
    assert torch.equal(got, beta.expand(3, cols))
