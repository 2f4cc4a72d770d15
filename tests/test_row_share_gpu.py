"""GPU parity of the row operators where several workgroups take a row together (row_any_kernel with SHARE 2 and 4): rows around the lines
of the choice, columns around its vectors, odd starts, in place.  Bars as for the other row kernels."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.util import NAME, TOL, as_f64, assert_close, to_dev

pytestmark = pytest.mark.gpu


def _run(op, x, g, b, out=None):
    from metalhlo_amd import kernels
    if op == "softmax":
        return kernels.softmax(x), oracle.softmax(as_f64(x))
    if op == "layer_norm":
        return kernels.layer_norm(x, g, b), oracle.layer_norm(as_f64(x), as_f64(g), as_f64(b), 1e-5)
    return kernels.rms_norm(x, g), oracle.rms_norm(as_f64(x), as_f64(g), 1e-5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=lambda d: NAME[d])
@pytest.mark.parametrize("op", ["softmax", "layer_norm", "rms_norm"])
@pytest.mark.parametrize("rows,cols", [(1, 8193), (64, 8209), (65, 16385), (128, 32769), (129, 9001), (9, 50257), (3, 65537), (127, 16383), (2, 131071)], ids=str)
def test_rows_in_shares(op, rows, cols, dtype):
    rng = np.random.default_rng(cols)
    x = to_dev(rng.standard_normal((rows, cols)) * 2 + 0.5, dtype)
    x[0, :] = 1.0                                       # a row of equal elements: no variance
    if cols > 100:
        x[-1, 7] = 60.0                                 # one that takes all of the softmax
    g, b = to_dev(1 + 0.1 * rng.standard_normal(cols), dtype), to_dev(0.1 * rng.standard_normal(cols), dtype)
    got, exp = _run(op, x, g, b)
    assert_close(got, exp, TOL[dtype], f"{op} {(rows, cols)}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=lambda d: NAME[d])
@pytest.mark.parametrize("op", ["softmax", "layer_norm", "rms_norm"])
@pytest.mark.parametrize("cols", [9001, 16385, 50257, 65537, 131071])
def test_same_bits_beside_any_rows(op, cols, dtype):
    """One, two and four workgroups a row add in the same order."""
    rng = np.random.default_rng(cols + 1)
    x = torch.randn(131, cols, device="cuda", generator=torch.Generator(device="cuda").manual_seed(cols)).to(dtype)
    g, b = to_dev(1 + 0.1 * rng.standard_normal(cols), dtype), to_dev(0.1 * rng.standard_normal(cols), dtype)
    from metalhlo_amd import kernels
    f = {"softmax": kernels.softmax, "layer_norm": lambda t: kernels.layer_norm(t, g, b), "rms_norm": lambda t: kernels.rms_norm(t, g)}[op]
    alone = f(x)
    for rows in (1, 64, 65, 128):
        assert torch.equal(f(x[:rows]), alone[:rows]), rows


def test_rows_in_place(lib):
    """y = x is one workgroup's business: the result of a call with a y of its own, bit for bit."""
    from metalhlo_amd import kernels
    x = torch.randn(17, 50257, device="cuda").bfloat16()
    want, y = kernels.softmax(x), x.clone()
    assert lib.mhip_softmax(torch.cuda.current_stream().cuda_stream, y.data_ptr(), y.data_ptr(), 17, 50257, kernels.DTYPE_CODE[torch.bfloat16]) == 0
    assert torch.equal(y, want)
