"""The output head of a short prompt against the product with the rounded table in 64 bits: groups of sixteen rows, blocks of
256, strips of sixteen columns (ragged, fewer than workgroups), k short of the 768 that a wave holds; GPT-2's use of it."""
import pytest
import torch

from metalhlo_amd import _lib, kernels

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 17, 128, 129, 256, 257, 512, 768])
@pytest.mark.parametrize("N,K", [(8, 768), (1000, 32), (4104, 736), (12360, 768)])
def test_head(dtype, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    # (guards: rows behind the table and in front of the result's end must not be read or written)
    w = torch.full((N + 16, K), float("nan"), device="cuda")
    w[:N] = torch.randn(N, K, generator=g, device="cuda") * K ** -0.5
    got = kernels.tied_head(x, w[:N])
    exp = x.double() @ w[:N].to(dtype).double().T.contiguous()
    assert got.shape == (M, N) and ((got.double() - exp).abs() <= EPS[dtype] * exp.abs().clamp(min=1.0)).all()


def test_values_that_are_not_finite_stay_in_their_place():
    x, w = torch.randn(70, 768, device="cuda").bfloat16(), torch.randn(1000, 768, device="cuda")
    w[333, 5], x[69, 700] = float("inf"), float("nan")
    got = kernels.tied_head(x, w)
    assert got[69].isnan().all() and not got[:69, 333].isfinite().any()
    got[:, 333] = 0
    assert got[:69].isfinite().all()


def test_refusals():
    bf = torch.bfloat16
    assert kernels.tied_head_served(768, 1000, 768, bf) and not kernels.tied_head_served(769, 1000, 768, bf)
    for n, k, dt in ((1000, 800, bf), (1000, 40, bf), (1001, 768, bf), (1000, 768, torch.float32)):
        assert not kernels.tied_head_served(4, n, k, dt)
        with pytest.raises((_lib.MhipError, TypeError)):
            kernels.tied_head(torch.zeros(4, k, dtype=dt, device="cuda"), torch.zeros(n, k, device="cuda"))


def test_matmul_of_129_to_192_rows_with_many_columns():
    """256-row tiles where their columns fill the device."""
    for M, N, K in ((129, 50304, 768), (192, 49400, 544)):
        g = torch.Generator(device="cuda").manual_seed(M)
        a, b = torch.randn(M, K, generator=g, device="cuda").bfloat16(), torch.randn(N, K, generator=g, device="cuda").bfloat16()
        got = kernels.matmul(a, b, trans_b=True)
        assert _lib.load().mhip_gemm_last_variant() == 2560
        rows = torch.arange(0, M, 7, device="cuda")
        exp = a[rows].float() @ b.float().T.contiguous()
        assert ((got[rows].float() - exp).abs() <= 2.0 ** -8 * exp.abs().clamp(min=K ** 0.5)).all()
