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
