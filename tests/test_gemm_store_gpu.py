"""GPU parity of the tile store of the 16-bit GEMM kernels (gemm_lds.h): rows of C off 16 bytes in chunks with what is left of a row element by element, fewer columns
than a chunk, the last column at the end of the tensor (what lies behind it stays), residuals that alias C.  Bounds as in test_gemm_few_tiles_gpu.py."""
import numpy as np
import pytest
import torch

from tests.test_gemm_few_tiles_gpu import _check
from tests.util import NAME, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("residual", [False, True], ids=["plain", "residual"])
@pytest.mark.parametrize("M,N,K", [(200, 1, 264), (193, 7, 128), (300, 9, 200), (257, 63, 264), (200, 65, 520), (513, 129, 96), (193, 1004, 1000), (700, 1001, 256)], ids=str)
@pytest.mark.parametrize("tb", [False, True], ids=["nn", "nt"])
def test_rows_of_any_alignment(M, N, K, tb, residual, dtype):
    _check(M, N, K, dtype, False, tb, residual)


def test_residual_that_is_the_result():
    from metalhlo_amd import kernels
    rng = np.random.default_rng(9)
    for M, N, K in ((300, 1001, 520), (260, 1000, 520), (4100, 777, 520)):
        a, b, r = (to_dev(rng.standard_normal(s), torch.bfloat16) for s in ((M, K), (K, N), (M, N)))
        want = kernels.matmul(a, b, residual=r)
        assert torch.equal(kernels.matmul(a, b, residual=r, out=r), want)
