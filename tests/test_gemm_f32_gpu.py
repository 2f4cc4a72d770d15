"""GPU parity of the fp32 GEMM kernels: the LDS ring of gemm_f32.hip (edges of its 64- and 128-wide tiles and 32-k
stages, split K, batches), the register-staged kernel for rows without 16-byte alignment, and blocks of rows in
gemm_skinny.hip.  Bound as in tests/test_gemm_few_tiles_gpu.py."""
import pytest
import torch

from tests.test_gemm_few_tiles_gpu import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)], ids=["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(60, 64, 36), (65, 16, 4), (68, 132, 132), (128, 768, 776), (193, 200, 31), (192, 2600, 100), (196, 64, 32), (200, 260, 1004), (513, 130, 67),
                                   (516, 132, 4100), (4100, 4092, 36)], ids=lambda v: str(v))
def test_f32(M, N, K, layout):
    _check(M, N, K, torch.float32, *layout, residual=N % 8 == 4)


def test_f32_batched():
    _check(100, 72, 68, torch.float32, False, False, True, batch=(5,))
    _check(260, 200, 132, torch.float32, True, True, True, batch=(3,))


def test_f32_views_at_odd_addresses():
    from metalhlo_amd import kernels
    M, N, K = 260, 264, 520
    a, b = torch.randn(M * K + 1, device="cuda")[1:].view(M, K), torch.randn(K * N + 1, device="cuda")[1:].view(K, N)
    got = kernels.matmul(a, b)
    e = a.double().cpu() @ b.double().cpu()
    fp32 = (K + 2) * 2.0 ** -24 * (a.double().cpu().abs() @ b.double().cpu().abs())
    assert ((got.double().cpu() - e).abs() <= fp32 + 2.0 ** -24 * (e.abs() + fp32)).all()


def test_f32_rows_do_not_depend_on_the_batch():
    """From 193 rows on, below a K of 4096, a row's sums are in one order whatever the number of rows."""
    from metalhlo_amd import kernels
    a, b = torch.randn(4608, 768, device="cuda"), torch.randn(768, 4096, device="cuda")
    big = kernels.matmul(a, b)
    assert torch.equal(kernels.matmul(a[:512].contiguous(), b), big[:512])
