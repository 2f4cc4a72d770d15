"""GPU parity of the few-row GEMM kernels whose weights land in LDS (gemm_strip.hip): edges of strips, of parts of K and of a
wave's share, and the count of arrivals in workspaces of any content (arrive.h).

Bound as in test_gemm_few_tiles_gpu.py: K 2^-24 of sum |a||b| for the fp32 sum, one rounding to the type, one more with a residual."""
import numpy as np
import pytest
import torch

from tests.test_gemm_few_tiles_gpu import ROUNDOFF, _check
from tests.util import NAME

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("M,N,K", [(1, 520, 1032), (16, 512, 1536), (9, 584, 1544), (17, 568, 2048), (32, 4104, 2056), (3, 8192, 4096), (8, 648, 8200), (32, 512, 16384)],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("tb", [False, True], ids=["nn", "nt"])
def test_parts(M, N, K, tb, dtype):
    _check(M, N, K, dtype, False, tb, residual=N % 16 == 8)


@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (16, 17, 64), (5, 33, 520), (8, 4096, 4096), (8, 47, 4088), (16, 31, 2048), (7, 16384, 512), (9, 100, 1016)], ids=lambda v: str(v))
def test_strips(M, N, K):
    _check(M, N, K, torch.bfloat16, False, True, residual=N % 2 == 1)


def test_strips_batched():
    _check(5, 40, 136, torch.float16, False, True, True, batch=(3,))


@pytest.mark.parametrize("tb", [False, True], ids=["nn", "nt"])
def test_workspace_of_any_content(lib, tb):
    """Counts left by nobody, by another launch, or all ones: the same bits, call after call, and a residual that aliases C is added once."""
    M, N, K = 12, 1000, 4104
    need = lib.mhip_gemm_workspace(M, N, K, 1, 0, int(tb), 3)
    assert need >= M * N * 4 * 9
    g = torch.Generator(device="cuda").manual_seed(3)
    a, b, r = (torch.randn(*s, generator=g, device="cuda").bfloat16() for s in ((M, K), (N, K) if tb else (K, N), (M, N)))
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    exact = a.double() @ (b.double().t() if tb else b.double())
    bound = K * 2.0 ** -24 * (a.double().abs() @ (b.double().abs().t() if tb else b.double().abs()))
    u = ROUNDOFF[torch.bfloat16]
    want = None
    for fill in (0, 255, 1, 128, None, None, None):
        if fill is not None:
            ws.fill_(fill)
        out = r.clone()
        rc = lib.mhip_gemm_ws(torch.cuda.current_stream().cuda_stream, a.data_ptr(), b.data_ptr(), None, out.data_ptr(), out.data_ptr(), M, N, K, 1, 0, 0, M * N, 0,
                              int(tb), 0, 3, ws.data_ptr(), need)
        assert rc == 0
        first = bound + u * (exact.abs() + bound)
        total = exact + r.double()
        assert ((out.double() - total).abs() <= first + u * (total.abs() + first)).all(), fill
        want = out if want is None else want
        assert torch.equal(out, want), fill
