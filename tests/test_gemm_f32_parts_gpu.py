"""fp32 products whose K is summed in parts: the same bits from workgroups of their own (with a workspace), from one that
takes the parts in turn (without), from 128-wide tiles and from rows that start on no 16-byte boundary, around the K
from which there are parts; values against float64 with the bound of tests/test_gemm_few_tiles_gpu.py."""
import pytest
import torch

from metalhlo_amd import _lib, kernels
from tests.test_gemm_few_tiles_gpu import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, False), (True, True)], ids=["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("M,N,K", [(193, 65, 511), (201, 130, 512), (333, 129, 769), (257, 63, 2049), (1025, 131, 1030), (194, 97, 33)], ids=lambda v: str(v))
def test_odd_rows(M, N, K, layout):
    _check(M, N, K, torch.float32, *layout, residual=M % 2 == 0)


@pytest.mark.parametrize("N,K", [(2048, 511), (2048, 600), (1000, 1536), (772, 3100), (130, 5000)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 1)])
def test_parts_have_the_bits_of_the_whole(N, K, ta, tb):
    lib, f32 = _lib.load(), kernels.DTYPE_CODE[torch.float32]
    g = torch.Generator(device="cuda").manual_seed(N + K)
    rows = 200
    x, w = torch.randn(8000, K, generator=g, device="cuda"), torch.randn(N * K + 1, generator=g, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream

    def product(M, odd, parts):
        a = (x[:M].t() if ta else x[:M]).contiguous()
        b = w[1:] if odd else w[1:].clone()
        out = torch.empty(M, N, device="cuda")
        n = lib.mhip_gemm_workspace(M, N, K, 1, ta, tb, f32) if parts else 0
        work = torch.empty(n, dtype=torch.uint8, device="cuda") if n else None
        assert lib.mhip_gemm_ws(stream, a.data_ptr(), b.data_ptr(), None, None, out.data_ptr(), M, N, K, 1, 0, 0, 0, ta, tb, 0, f32,
                                work.data_ptr() if n else None, n) == 0
        return out, n

    whole, _ = product(rows, False, False)
    split, n = product(rows, False, True)
    assert (n > 0) == (K >= 512) and torch.equal(split, whole)
    assert torch.equal(product(rows, True, True)[0], whole)
    assert torch.equal(product(8000, False, True)[0][:rows], whole)


@pytest.mark.parametrize("M,N,K", [(33, 2336, 20), (48, 3104, 132), (100, 1568, 516), (65, 2336, 36), (128, 3104, 772), (192, 800, 1028), (128, 2304, 3072), (48, 3068, 132)], ids=lambda v: str(v))
def test_strips_of_48_columns(M, N, K):
    """Few-row products whose strips are three columns a lane, the last strip ragged."""
    _check(M, N, K, torch.float32, False, False, residual=M % 2 == 0)


@pytest.mark.parametrize("M,N,K,tb", [(33, 2304, 1025, True), (48, 2303, 1024, False), (100, 767, 3073, True), (192, 101, 1030, False), (32, 767, 1025, True)], ids=lambda v: str(v))
def test_few_rows_off_16_bytes(M, N, K, tb):
    _check(M, N, K, torch.float32, False, tb, residual=M % 2 == 0)


@pytest.mark.parametrize("M,N,K,tb", [(33, 768, 2048, False), (48, 772, 3076, False), (128, 768, 3072, False), (100, 512, 2052, False), (64, 1024, 4096, True),
                                      (128, 511, 2047, True), (128, 1024, 4096, False)], ids=lambda v: str(v))
def test_few_rows_with_blocks_and_parts_chosen_together(M, N, K, tb):
    _check(M, N, K, torch.float32, False, tb, residual=M % 8 == 0)


@pytest.mark.parametrize("M,N,K", [(3970, 3972, 36), (3969, 3972, 516)], ids=lambda v: str(v))
def test_large_products_off_16_bytes_have_the_bits_of_aligned_ones(M, N, K):
    """Tiles of 64x64 with four-byte loads where an aligned product has 128x128."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N * K + 1, generator=g, device="cuda")
    assert torch.equal(kernels.matmul(a, w[1:].view(K, N)), kernels.matmul(a, w[1:].clone().view(K, N)))


@pytest.mark.parametrize("ta", [False, True])
def test_twelve_columns_keep_a_rows_bits(ta):
    """The narrowest C whose rows have the same bits from 193 rows on."""
    g = torch.Generator(device="cuda").manual_seed(12)
    a, b = torch.randn(4000, 1030, generator=g, device="cuda"), torch.randn(1030, 12, generator=g, device="cuda")

    def rows(n):
        x = (a[:n].t() if ta else a[:n]).contiguous()
        return kernels.matmul(x, b, trans_a=ta)[:193]
    assert torch.equal(rows(193), rows(4000))


@pytest.mark.parametrize("M,N,K", [(64, 4096, 4096), (33, 4100, 4096), (52, 8192, 3264)], ids=lambda v: str(v))
def test_few_rows_whose_sums_take_all_of_64_kb(M, N, K):
    """Strips of 32 columns by 64 rows in parts of K: the waves' sums fill what a launch gets without asking for more."""
    _check(M, N, K, torch.float32, False, False, residual=M % 2 == 0)
