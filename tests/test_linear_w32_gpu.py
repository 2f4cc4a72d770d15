"""Linear layers with fp32 parameters (mhip_linear_w32, mhip_finish_norm) against the same sums in 64 bits over the
parameters rounded to the compute type, at the edges of their strips (16 columns), row groups (16, 64) and k steps
(32, 24 of them held at once)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _draw(seed, *shape, scale=1.0, shift=0.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, generator=g, device="cuda") * scale + shift


def _gelu(v):
    return 0.5 * v * (1 + torch.tanh(0.7978845608028654 * (v + 0.044715 * v ** 3)))


def _close(got, exp, scale, roundings):
    """One half unit per rounding of the result to its type, and the fp32 sums (K terms, each side 2^-24)."""
    assert torch.isfinite(got).all()
    err = (got.double() - exp).abs()
    assert (err <= roundings * EPS[got.dtype] * exp.abs().clamp(min=scale) + 1e-6 * scale).all(), float(err.max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 16, 17, 37, 64, 65, 192])
@pytest.mark.parametrize("N,K,trans_b", [(8, 8, False), (24, 776, False), (200, 768, False), (136, 1000, False),
                                         (8, 16, True), (1000, 768, True), (40, 1000, True), (8208, 64, True)])
def test_linear(dtype, M, N, K, trans_b):
    from metalhlo_amd import kernels
    x = _draw(1, M, K).to(dtype)
    w = _draw(2, *((N, K) if trans_b else (K, N)), scale=K ** -0.5)
    b, r = _draw(3, N, scale=0.5), _draw(4, M, N).to(dtype)
    w64 = w.to(dtype).double()
    s = x.double() @ (w64.T.contiguous() if trans_b else w64)
    ahead = (_draw(5, 64, 136), _draw(6, 24, 8))          # (a hint: never part of the result)
    _close(kernels.linear(x, w, trans_b=trans_b), s, 1.0, 1)
    _close(kernels.linear(x, w, b, "gelu", trans_b, ahead=ahead), _gelu(s + b.to(dtype).double()), 1.0, 1)
    # the sum is rounded, and rounded again behind the residual
    _close(kernels.linear(x, w, b, trans_b=trans_b, residual=r), s + b.to(dtype).double() + r.double(), 4.0, 2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(1, 64, 200), (37, 768, 3072), (65, 1032, 768), (192, 4096, 136)])
@pytest.mark.parametrize("parts", [0, 1, 3, 8])
def test_parts_and_finish_norm(dtype, M, N, K, parts):
    """Shares of K, some of them empty where there are more parts than steps, and the LayerNorm behind their sum."""
    from metalhlo_amd import kernels
    x, w, b, r = _draw(1, M, K).to(dtype), _draw(2, K, N, scale=K ** -0.5), _draw(3, N, scale=0.5), _draw(4, M, N).to(dtype)
    g, be = _draw(5, N, scale=0.1, shift=1.0), _draw(6, N, scale=0.1)
    sums = kernels.linear(x, w, parts=parts) if parts else None
    c, h = kernels.finish_norm(sums, b if parts else None, r, (g, be, 1e-5))
    if parts:
        assert sums.shape == (parts, M, N)
        s = x.double() @ w.to(dtype).double()
        assert (sums.double().sum(0) - s).abs().max() <= 1e-5 * s.abs().max()
        _close(c, s + b.to(dtype).double() + r.double(), 4.0, 2)
    else:
        assert torch.equal(c, r)
    c64 = c.double()
    n = (c64 - c64.mean(-1, keepdim=True)) / (c64.var(-1, unbiased=False, keepdim=True) + 1e-5).sqrt()
    _close(h, n * g.to(dtype).double() + be.to(dtype).double(), 1.0, 1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N", [24, 40, 200, 768, 1000, 3080, 4096])
def test_rows_of_equal_elements_have_no_variance(dtype, N):
    """The sum of N equal elements of up to 11 bits is exact, so is its quotient by N: nothing is left in front of beta."""
    from metalhlo_amd import kernels
    v = torch.cat([torch.arange(1, 200, device="cuda") / 16, torch.linspace(300, 2000, 57, device="cuda")]).to(dtype)
    x, g, b = v[:, None].repeat(1, N), _draw(1, N, shift=1.0), _draw(2, N)
    for beta in (b, torch.zeros(N, device="cuda")):
        _, h = kernels.finish_norm(None, None, x, (g, beta, 1e-12))
        assert torch.equal(h, beta.to(dtype).expand_as(h))


def test_refusals():
    from metalhlo_amd import _lib, kernels
    bf = torch.bfloat16
    assert kernels.linear_served(192, 768, 768, bf) and not kernels.linear_served(193, 768, 768, bf)
    for n, k, dt in ((766, 768, bf), (768, 770, bf), (768, 768, torch.float32)):
        assert not kernels.linear_served(4, n, k, dt)
        with pytest.raises((_lib.MhipError, TypeError)):
            kernels.linear(torch.zeros(4, k, dtype=dt, device="cuda"), torch.zeros(k, n, device="cuda"))
    with pytest.raises(_lib.MhipError):
        kernels.linear(torch.zeros(4, 64, dtype=bf, device="cuda"), torch.zeros(64, 64, device="cuda"), parts=9)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S", [(1, 1), (2, 37), (3, 64)])
def test_gpt2_prompt_matches_the_converted_parameters(dtype, B, S):
    """The short-prompt form of GPT-2 against the form for more tokens: the same roundings, fp32 sums in another order.  Where
    those differ a value rounds the other way and carries on, at most a few units by the second layer."""
    from metalhlo_amd.gpt2 import GPT2, GPT2Config, init_params
    cfg = GPT2Config(n_layer=2, d_model=256, n_head=4, d_ff=1024, vocab=1000, n_pos=64)
    model = GPT2(cfg, init_params(cfg, seed=3), compute_dtype=dtype)
    ids = torch.randint(0, cfg.vocab, (B, S), generator=torch.Generator().manual_seed(1), dtype=torch.int32).cuda()
    assert model._few_tokens(B * S)
    few = model.forward(ids)
    model._few_tokens = lambda tokens: False
    many = model.forward(ids)
    assert few.shape == many.shape == (B, S, cfg.vocab)
    err = (few.double() - many.double()).norm() / many.double().norm()
    assert err <= 2 * EPS[dtype], float(err)
