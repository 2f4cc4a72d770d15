"""GPU parity of attention and its projection in one launch with four heads a part: what 16 and more heads take, the most LDS and all waves at the product; and of a model whose layers
take it.  Bounds as in test_attend_project_gpu.py and test_gemm_sums_gpu.py."""
import numpy as np
import pytest
import torch

from tests.util import NAME, to_dev

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("B,S,H,N,parts", [(1, 64, 16, 1024, 4), (2, 32, 16, 264, 4), (1, 33, 20, 1280, 5), (1, 37, 32, 72, 8), (2, 1, 16, 8, 4), (1, 32, 28, 40, 7)], ids=str)
def test_sums_of_four_heads(B, S, H, N, parts, dtype):
    from metalhlo_amd import kernels
    assert kernels.attend_project_served(B, S, H, 64, N, dtype)
    rng = np.random.default_rng(B * 1000 + S + N)
    qkv = to_dev(rng.standard_normal((B * S, 3 * H * 64)), dtype)
    w = to_dev(rng.standard_normal((H * 64, N)), torch.float32)
    sums = kernels.attend_project(qkv, w, B, H, ahead=(to_dev(rng.standard_normal((64, 128)), torch.float32),))
    assert sums.dtype == torch.float32 and sums.shape == (parts, B * S, N)
    x, r = kernels.causal_attention(qkv, B, H).double(), w.to(dtype).double()
    for p, heads in enumerate(torch.arange(H * 64, device="cuda").chunk(parts)):        # each part is the product of its heads
        error = (sums[p].double() - x[:, heads] @ r[heads]).abs()
        assert bool((error <= len(heads) * 2.0 ** -23 * (x[:, heads].abs() @ r[heads].abs())).all()), (p, float(error.max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("d_model,n_head", [(768, 12), (1024, 16)])
@pytest.mark.parametrize("B,S", [(1, 37), (2, 20), (1, 64), (2, 32)])
def test_gpt2_prompt_forms_agree(B, S, d_model, n_head, dtype):
    """33 to 64 tokens, whose layers take attention and projection together, against the form for many tokens: the same roundings, fp32 sums in
    another order."""
    from metalhlo_amd import kernels
    from metalhlo_amd.gpt2 import GPT2, GPT2Config, init_params
    cfg = GPT2Config(n_layer=2, d_model=d_model, n_head=n_head, d_ff=4 * d_model, vocab=1000)
    model = GPT2(cfg, init_params(cfg, seed=3), compute_dtype=dtype)
    ids = torch.randint(0, cfg.vocab, (B, S), generator=torch.Generator().manual_seed(1), dtype=torch.int32).cuda()
    assert model._few_tokens(B * S) and kernels.attend_project_served(B, S, n_head, 64, d_model, dtype)
    assert not kernels.linear_norm_served(B * S, d_model, d_model, dtype)
    few = model.forward(ids)
    model._few_tokens, model._full_tiles = (lambda tokens: False), 0
    many = model.forward(ids)
    err = (few.double() - many.double()).norm() / many.double().norm()
    assert err <= 2 * EPS[dtype], float(err)
