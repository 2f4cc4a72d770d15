"""GPU parity of the 16-bit GEMM for operands without vector alignment (gemm_any.hip): sizes around its 64- and
128-wide tiles, its 64-k stages and the eight-element pieces, views at odd addresses, split K, batches; results
against float64 with the bound of tests/test_gemm_few_tiles_gpu.py."""
import numpy as np
import pytest
import torch

from tests.test_gemm_few_tiles_gpu import _check
from tests.util import NAME, as_f64, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)], ids=["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(1, 3, 5), (3, 1, 1), (65, 7, 9), (65, 129, 63), (127, 66, 65), (193, 130, 127), (200, 515, 129), (129, 333, 1031), (515, 257, 4099),
                                   (2049, 2047, 67), (2047, 2100, 130)], ids=lambda v: str(v))
def test_any_size(M, N, K, layout, dtype):
    _check(M, N, K, dtype, *layout, residual=N % 2 == 1)


def test_any_batched():
    _check(67, 201, 133, torch.bfloat16, False, False, True, batch=(5,))
    _check(130, 77, 45, torch.float16, True, True, True, batch=(3,))


@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)], ids=["nn", "tt"])
def test_views_at_odd_addresses(ta, tb):
    """Aligned sizes, operands, bias, residual and result that start two bytes behind an aligned address."""
    from metalhlo_amd import kernels
    M, N, K = 200, 264, 520
    rng = np.random.default_rng(3)

    def odd(*shape):
        flat = to_dev(rng.standard_normal(int(np.prod(shape)) + 1), torch.bfloat16)
        return flat[1:].view(*shape)
    a, b = odd(*((K, M) if ta else (M, K))), odd(*((N, K) if tb else (K, N)))
    bias, res, out = odd(N), odd(M, N), odd(M, N)
    kernels.matmul(a, b, bias=bias, residual=res, trans_a=ta, trans_b=tb, out=out)
    A, B = (as_f64(a).T if ta else as_f64(a)), (as_f64(b).T if tb else as_f64(b))
    e = A @ B + as_f64(bias)
    fp32 = (K + 2) * 2.0 ** -24 * (np.abs(A) @ np.abs(B) + np.abs(as_f64(bias)))
    bound = fp32 + 2.0 ** -8 * (np.abs(e) + fp32)
    e = e + as_f64(res)
    assert np.all(np.abs(as_f64(out) - e) <= bound + 2.0 ** -8 * (np.abs(e) + bound))

