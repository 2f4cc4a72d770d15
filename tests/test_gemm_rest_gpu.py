"""The 128x192 tile where K is no multiple of its 32-k stages and both operands have k as the slow axis: the rest of K in one
stage behind the loop, alone and in the last part of a split K.  Bits of the 128-row tiles; 64-bit values."""
import pytest
import torch

from metalhlo_amd import _lib, kernels

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(2056, 2328, 33), (2056, 2328, 47), (3080, 1544, 48), (2568, 2120, 63), (2056, 4616, 545), (768, 3072, 1001)])
def test_rest_of_k(dtype, M, N, K, monkeypatch):
    g = torch.Generator(device="cuda").manual_seed(K)
    # (a guard behind the operands: what lies past K must not be multiplied)
    a = torch.full((K + 40, M), float("nan"), dtype=dtype, device="cuda")
    b = torch.full((K + 40, N), float("nan"), dtype=dtype, device="cuda")
    a[:K], b[:K] = torch.randn(K, M, generator=g, device="cuda").to(dtype), torch.randn(K, N, generator=g, device="cuda").to(dtype)
    bias, res = torch.randn(N, generator=g, device="cuda").to(dtype), torch.randn(M, N, generator=g, device="cuda").to(dtype)
    got = {}
    for tile in ("2569", "128"):
        monkeypatch.setenv("MHIP_GEMM_TILE", tile)
        got[tile] = kernels.matmul(a[:K], b[:K], bias, "relu", trans_a=True, residual=res)
        if M > 768:
            assert _lib.load().mhip_gemm_last_variant() == int(tile)
    assert torch.equal(got["2569"], got["128"])
    exp = torch.relu(a[:K].double().T.contiguous() @ b[:K].double() + bias.double())
    scale = exp.abs().clamp(min=K ** 0.5)
    assert ((got["2569"].double() - exp - res.double()).abs() <= 2 * EPS[dtype] * (scale + res.double().abs())).all()


@pytest.mark.parametrize("M,N,K", [(768, 3072, 8200), (512, 1000, 16383), (640, 768, 4097)])
def test_rest_of_a_split_k(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.randn(K, n, generator=g, device="cuda").bfloat16() for n in (M, N))
    got = kernels.matmul(a, b, trans_a=True)
    exp = a.double().T.contiguous() @ b.double()
    assert ((got.double() - exp).abs() <= EPS[torch.bfloat16] * exp.abs().clamp(min=K ** 0.5)).all()
    # the last k alone decides: a rest that is left out, or taken twice, shows
    a[:-1].zero_()
    last = kernels.matmul(a, b, trans_a=True)
    assert torch.equal(last, (a[-1].float()[:, None] * b[-1].float()[None]).bfloat16())
