"""GPU parity of linear layers that normalise their rows, and of those whose last workgroup adds the parts of K up (linear_w32.hip): groups of 16
rows, the end of a wave's share, workspaces of any content.  Bounds: a product of K terms summed in fp32 is off by at most K 2^-24 of sum |a||b|, one
rounding to the type, one more with a residual; LayerNorm's rounding to the type moves each operand by one unit of its last place."""
import numpy as np
import pytest
import torch

from tests.util import NAME, as_f64, to_dev

pytestmark = pytest.mark.gpu
ROUNDOFF = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _params(rng, K, N):
    f32 = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda()  # noqa: E731
    return f32(K, N) * K ** -0.5, f32(N), 1 + 0.1 * f32(K), 0.1 * f32(K)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (16, 40, 64), (17, 2304, 768), (32, 768, 760), (5, 72, 200), (31, 8, 520)], ids=str)
def test_normalised_rows(M, N, K, dtype):
    from metalhlo_amd import kernels
    rng = np.random.default_rng(K + M)
    x = to_dev(rng.standard_normal((M, K)) * 2 + 0.7, dtype)
    x[0] = 3.0                                           # a row of equal elements: no variance
    w, bias, gamma, beta = _params(rng, K, N)
    assert kernels.linear_norm_served(M, N, K, dtype)
    got = as_f64(kernels.linear_layer(x, w, bias, "relu", norm=(gamma, beta, 1e-5)))
    r = lambda t: as_f64(t.to(dtype))  # noqa: E731
    v = as_f64(x)
    h = (v - v.mean(1, keepdims=True)) / np.sqrt(v.var(1, keepdims=True) + 1e-5) * r(gamma) + r(beta)
    u, W = ROUNDOFF[dtype], np.abs(r(w))
    e = np.maximum(h @ r(w) + r(bias), 0)
    bound = (u + (K + 8) * 2.0 ** -24) * (np.abs(h) + 1e-4) @ W + 2.0 ** -22 * np.abs(r(bias))
    assert np.all(np.abs(got - e) <= bound + u * (np.abs(e) + bound)), (M, N, K)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("M,N,K", [(1, 768, 3072), (16, 64, 1160), (17, 136, 6144), (32, 768, 3064), (9, 8, 9000)], ids=str)
def test_parts_added_up_in_one_launch(lib, M, N, K, dtype):
    from metalhlo_amd import kernels
    rng = np.random.default_rng(K)
    x, res = to_dev(rng.standard_normal((M, K)), dtype), to_dev(rng.standard_normal((M, N)), dtype)
    w, bias, _, _ = _params(rng, K, N)
    need, code = lib.mhip_linear_w32_workspace(M, N, K), kernels.DTYPE_CODE[dtype]
    assert need > 0
    ws, want = torch.empty(need, dtype=torch.uint8, device="cuda"), None
    A, W, b, u = as_f64(x), as_f64(w.to(dtype)), as_f64(bias.to(dtype)), ROUNDOFF[dtype]
    first = A @ W + b
    bound = (K + 8) * 2.0 ** -24 * (np.abs(A) @ np.abs(W) + np.abs(b))
    bound = bound + u * (np.abs(first) + bound)
    e = first + as_f64(res)
    bound = bound + u * (np.abs(e) + bound)
    for fill in (0, 255, 128, None, None):
        if fill is not None:
            ws.fill_(fill)
        c = torch.full_like(res, float("nan"))
        assert lib.mhip_linear_w32_layer(torch.cuda.current_stream().cuda_stream, x.data_ptr(), None, None, 0.0, w.data_ptr(), bias.data_ptr(), res.data_ptr(), c.data_ptr(),
                                         M, N, K, 0, code, ws.data_ptr(), need, 0, None) == 0
        assert np.all(np.abs(as_f64(c) - e) <= bound), (M, N, K, fill)
        want = c if want is None else want
        assert torch.equal(c, want), fill
    assert torch.equal(kernels.linear_layer(x, w, bias, residual=res), want)


@pytest.mark.parametrize("B,S", [(1, 1), (1, 16), (2, 16), (3, 5)], ids=str)
def test_gpt2_layers_with_and_without_their_norms(B, S, monkeypatch):
    """A prompt of few tokens through both forms of the layers: the same intermediates rounded to 16 bits, sums in another order."""
    from metalhlo_amd import kernels
    from metalhlo_amd.gpt2 import GPT2, GPT2Config, init_params
    cfg = GPT2Config(n_layer=3, d_model=256, n_head=4, d_ff=1600, vocab=640, n_pos=64)
    model = GPT2(cfg, init_params(cfg), torch.float16)
    ids = torch.randint(0, cfg.vocab, (B, S), device="cuda", dtype=torch.int32)
    got = model.forward(ids).double()
    monkeypatch.setattr(kernels, "linear_norm_served", lambda *a: False)
    want = model.forward(ids).double()
    assert (got - want).norm() <= 4e-3 * want.norm()     # (perf tolerance of a network in f16: every intermediate rounded once)
